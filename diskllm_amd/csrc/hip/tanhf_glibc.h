/*
 * tanhf_glibc.h -- bit-exact restatement of the host libm tanhf() that the
 * reference's logit soft-capping calls (src/core/context.c:604-606 after a
 * prefill, :873-876 after a decode step: logits[i] = cap * tanhf(logits[i] / cap)).
 *
 * Third-party dependency: GNU C Library 2.35 (Ubuntu 2.35-0ubuntu3.11), functions
 * tanhf (sysdeps/ieee754/flt-32/s_tanhf.c) and the expm1f it calls
 * (sysdeps/ieee754/flt-32/s_expm1f.c).  Both are the published fdlibm float
 * algorithms (Sun Microsystems, 1993; float conversion by Ian Lance Taylor):
 *   tanh(x) = sign(x) * (1 - 2 / (expm1(2|x|) + 2))   for 1 <= |x| < 22,
 *           = sign(x) * (-t / (t + 2)), t = expm1(-2|x|)  for 2^-55 <= |x| < 1,
 *           = x * (1 + x) below, sign(x) * 1 at and above 22;
 *   expm1(x): k = round(x / ln2), r = x - k ln2 split into hi + lo with a
 *   correction c, then expm1(r) from the rational form
 *   r - (r * e - r^2/2), R1 = 1 + r^2/2 * (Q1 + ... + Q5 (r^2/2)^4), and the
 *   result rescaled by 2^k with the per-k cases of the algorithm.
 * Every operation is one IEEE float operation in source order (x86-64 SSE, no
 * contraction), which is what the hipcc flags of this library give on the GPU
 * (-ffp-contract=off, correctly rounded float division, denormals kept).  The
 * constants are the algorithm's published float constants, written as bit
 * patterns.
 *
 * Usable on the host (gcc) and the device (hipcc).
 */
#ifndef DLK_TANHF_GLIBC_H
#define DLK_TANHF_GLIBC_H

#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define DLK_TH __host__ __device__ __forceinline__
#else
#define DLK_TH static inline
#endif

DLK_TH float dlk_th_u2f(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
DLK_TH uint32_t dlk_th_f2u(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

/* expm1f for the arguments tanhf passes: finite, |x| < 44. */
DLK_TH float dlk_expm1f_glibc(float x) {
    const float kLn2Hi = dlk_th_u2f(0x3f317180u), kLn2Lo = dlk_th_u2f(0x3717f7d1u);
    const float kInvLn2 = dlk_th_u2f(0x3fb8aa3bu);
    const float kQ1 = dlk_th_u2f(0xbd088889u), kQ2 = dlk_th_u2f(0x3ad00d01u), kQ3 = dlk_th_u2f(0xb8a670cdu),
                kQ4 = dlk_th_u2f(0x36867e54u), kQ5 = dlk_th_u2f(0xb457edbbu);
    const uint32_t ux = dlk_th_f2u(x);
    const int neg = (ux >> 31) != 0;
    const uint32_t ax = ux & 0x7fffffffu;
    if (ax >= 0x4195b844u && neg) return -1.0f;       /* x <= -27 ln2 (the huge-x cases do not occur) */
    float hi, lo, c = 0.0f;
    int k;
    if (ax > 0x3eb17218u) {                            /* |x| > ln2 / 2: reduce */
        if (ax < 0x3f851592u) {                        /* |x| < 1.5 ln2 */
            if (!neg) { hi = x - kLn2Hi; lo = kLn2Lo; k = 1; }
            else { hi = x + kLn2Hi; lo = -kLn2Lo; k = -1; }
        } else {
            k = (int)(kInvLn2 * x + (neg ? -0.5f : 0.5f));
            const float t = (float)k;
            hi = x - t * kLn2Hi;                       /* exact */
            lo = t * kLn2Lo;
        }
        x = hi - lo;
        c = (hi - x) - lo;
    } else if (ax < 0x33000000u) {                     /* |x| < 2^-25 */
        return x;
    } else {
        k = 0;
    }
    const float hfx = 0.5f * x;
    const float hxs = x * hfx;
    const float r1 = 1.0f + hxs * (kQ1 + hxs * (kQ2 + hxs * (kQ3 + hxs * (kQ4 + hxs * kQ5))));
    float t = 3.0f - r1 * hfx;
    float e = hxs * ((r1 - t) / (6.0f - x * t));
    if (k == 0) return x - (x * e - hxs);
    e = (x * (e - c) - c);
    e -= hxs;
    if (k == -1) return 0.5f * (x - e) - 0.5f;
    if (k == 1) {
        if (x < -0.25f) return -2.0f * (e - (x + 0.5f));
        return 1.0f + 2.0f * (x - e);
    }
    float y;
    if (k <= -2 || k > 56) {
        y = 1.0f - (e - x);
        y = dlk_th_u2f(dlk_th_f2u(y) + ((uint32_t)k << 23));
        return y - 1.0f;
    }
    if (k < 23) {
        t = dlk_th_u2f(0x3f800000u - (0x1000000u >> k));   /* 1 - 2^-k */
        y = t - (e - x);
    } else {
        t = dlk_th_u2f((uint32_t)(0x7f - k) << 23);         /* 2^-k */
        y = x - (e + t);
        y += 1.0f;
    }
    return dlk_th_u2f(dlk_th_f2u(y) + ((uint32_t)k << 23));
}

/* tanhf, bit-identical to glibc 2.35 tanhf on x86-64 (NaN inputs give a NaN). */
DLK_TH float dlk_tanhf_glibc(float x) {
    const uint32_t ux = dlk_th_f2u(x);
    const uint32_t ax = ux & 0x7fffffffu;
    const int neg = (ux >> 31) != 0;
    if (ax >= 0x7f800000u) {
        if (ax > 0x7f800000u) return x + x;            /* NaN */
        return neg ? -1.0f : 1.0f;                     /* 1/x +- 1 at +-inf */
    }
    float z;
    if (ax < 0x41b00000u) {                            /* |x| < 22 */
        if (ax == 0) return x;                         /* +-0 */
        if (ax < 0x24000000u) return x * (1.0f + x);   /* |x| < 2^-55 */
        const float a = dlk_th_u2f(ax);
        if (ax >= 0x3f800000u) {                       /* |x| >= 1 */
            const float t = dlk_expm1f_glibc(2.0f * a);
            z = 1.0f - 2.0f / (t + 2.0f);
        } else {
            const float t = dlk_expm1f_glibc(-2.0f * a);
            z = -t / (t + 2.0f);
        }
    } else {
        z = 1.0f;                                      /* 1 - tiny rounds to 1 */
    }
    return neg ? -z : z;
}

/* The reference's soft-cap of one logit: cap * tanhf(x / cap). */
DLK_TH float dlk_softcap_glibc(float x, float cap) { return cap * dlk_tanhf_glibc(x / cap); }

/* ---- the same for the common range, branch-free --------------------------------
 * For q = |x / cap| in [2^-60, 0.75 ln2) tanhf takes -t / (t + 2) with
 * t = expm1f(-2 q), and that takes k = 0 (2 q <= ln2 / 2) or k = -1: two forms
 * that differ by a constant and a final scaling, so both are computed without a
 * branch (with k = 0 the correction c is 0 and x * (e - c) - c is x * e; below
 * 2^-25, where expm1f returns its argument, x + x^2 / 2 rounds to x).  Every
 * operation keeps its value and its order; what is left out is the divisions'
 * scaling for operands near the ends of the exponent range, which do not occur:
 * the 80 vector instructions of the general form are about 60. */

/* n / d correctly rounded, for normal n, d and quotient well inside the exponent
 * range: the division sequence of the hardware without its scaling and fix-up
 * (reciprocal, one Newton step, quotient, two remainder corrections). */
DLK_TH float dlk_div_inner(float n, float d) {
#if defined(__HIP_DEVICE_COMPILE__)
    const float y0 = __builtin_amdgcn_rcpf(d);
#else
    const float y0 = 1.0f / d;
#endif
    const float y = __builtin_fmaf(__builtin_fmaf(-d, y0, 1.0f), y0, y0);
    const float q0 = n * y;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-d, q0, n), y, q0);
    return __builtin_fmaf(__builtin_fmaf(-d, q1, n), y, q1);
}

/* What the caps need of cap: its reciprocal rounded to float, with which two
 * remainder corrections round x / cap correctly (Markstein's theorem: a
 * correctly rounded reciprocal of a divisor whose significand is not all ones),
 * or 0 where that is not given and the general form is taken. */
DLK_TH float dlk_softcap_recip(float cap) {
    const uint32_t u = dlk_th_f2u(cap);
    if (!(cap >= 0x1p-20f && cap <= 0x1p40f) || (u & 0x7fffffu) == 0x7fffffu) return 0.0f;
    return (float)(1.0 / (double)cap);
}

/* |x / cap| (recip from dlk_softcap_recip; meaningful where dlk_softcap_common holds) */
DLK_TH float dlk_softcap_quot(float x, float cap, float recip) {
    const float a = __builtin_fabsf(x);
    const float q0 = a * recip;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-cap, q0, a), recip, q0);
    return __builtin_fmaf(__builtin_fmaf(-cap, q1, a), recip, q1);
}

/* q's place above the lower end of the common range; the form below holds where
 * this is under DLK_SOFTCAP_SPAN (unsigned: NaN, 0 and everything outside is not). */
#define DLK_SOFTCAP_SPAN (0x3f051592u - 0x21800000u)
DLK_TH uint32_t dlk_softcap_place(float q) { return dlk_th_f2u(q) - 0x21800000u; }

/* cap * tanhf(x / cap) for q = |x / cap| in the common range. */
DLK_TH float dlk_softcap_common(float x, float q, float cap) {
    const float kLn2Hi = dlk_th_u2f(0x3f317180u), kLn2Lo = dlk_th_u2f(0x3717f7d1u);
    const float kQ1 = dlk_th_u2f(0xbd088889u), kQ2 = dlk_th_u2f(0x3ad00d01u), kQ3 = dlk_th_u2f(0xb8a670cdu),
                kQ4 = dlk_th_u2f(0x36867e54u), kQ5 = dlk_th_u2f(0xb457edbbu);
    const float x2 = -2.0f * q;
    const int low = -x2 > dlk_th_u2f(0x3eb17218u);     /* k = -1 */
    const float hi = x2 + (low ? kLn2Hi : 0.0f);
    const float lo = low ? -kLn2Lo : 0.0f;
    const float r = hi - lo;
    const float c = (hi - r) - lo;
    const float hfx = 0.5f * r;
    const float hxs = r * hfx;
    const float r1 = 1.0f + hxs * (kQ1 + hxs * (kQ2 + hxs * (kQ3 + hxs * (kQ4 + hxs * kQ5))));
    const float t = 3.0f - r1 * hfx;
    float e = hxs * dlk_div_inner(r1 - t, 6.0f - r * t);
    e = r * (e - c) - c;
    e -= hxs;
    const float y0 = r - e;
    const float y = low ? 0.5f * y0 - 0.5f : y0;
    return __builtin_copysignf(cap * dlk_div_inner(-y, y + 2.0f), x);
}

/* ---- and for all but a few values, branch-free ----------------------------------
 * q in [2^-60, 7.75): expm1f's argument is -2 q below 1 and 2 q from there on, and
 * k is one of 0, -1, -2, -3 or 3 .. 22, so every per-k form is (A + d) 2^k - B with
 * d = r - e: A is 1 - 2^-k from k = 3 on, 1 at k = -2 and -3, else 0; B is 1 at
 * k = -2 and -3, 1/2 at k = -1, else 0 (adding or subtracting 0 and scaling by a
 * power of two change nothing).  The two special ranges of the reduction give the
 * same k and the same hi, lo and c as its general form there.  x = 0 comes out as
 * 0, and from 16 cap on tanhf is 1 (its 1 - 2 / (t + 2) rounds to 1 from q = 9.02). */
#define DLK_SOFTCAP_WIDE_SPAN (0x40f80000u - 0x21800000u)
#define DLK_SOFTCAP_ONE 16.0f

/* Whether dlk_softcap_wide holds for x (q = dlk_softcap_quot of it; cap16 = 16 cap). */
DLK_TH int dlk_softcap_wide_ok(float x, float q, float cap16) {
    return (dlk_softcap_place(q) < DLK_SOFTCAP_WIDE_SPAN) | (x == 0.0f) | (__builtin_fabsf(x) >= cap16);
}

/* cap * tanhf(x / cap) where dlk_softcap_wide_ok. */
DLK_TH float dlk_softcap_wide(float x, float q, float cap, float cap16) {
    const float kLn2Hi = dlk_th_u2f(0x3f317180u), kLn2Lo = dlk_th_u2f(0x3717f7d1u);
    const float kInvLn2 = dlk_th_u2f(0x3fb8aa3bu);
    const float kQ1 = dlk_th_u2f(0xbd088889u), kQ2 = dlk_th_u2f(0x3ad00d01u), kQ3 = dlk_th_u2f(0xb8a670cdu),
                kQ4 = dlk_th_u2f(0x36867e54u), kQ5 = dlk_th_u2f(0xb457edbbu);
    const int one = __builtin_fabsf(x) >= cap16;
    q = one ? 1.0f : q;                                /* (any value of the range) */
    const int neg = q < 1.0f;
    const float x2 = neg ? -2.0f * q : 2.0f * q;
    const int k = (int)(kInvLn2 * x2 + (neg ? -0.5f : 0.5f));
    const float kf = (float)k;
    const float hi = x2 - kf * kLn2Hi;
    const float lo = kf * kLn2Lo;
    const float r = hi - lo;
    const float c = (hi - r) - lo;
    const float hfx = 0.5f * r;
    const float hxs = r * hfx;
    const float r1 = 1.0f + hxs * (kQ1 + hxs * (kQ2 + hxs * (kQ3 + hxs * (kQ4 + hxs * kQ5))));
    const float t = 3.0f - r1 * hfx;
    float e = hxs * dlk_div_inner(r1 - t, 6.0f - r * t);
    e = r * (e - c) - c;
    e -= hxs;
    const float A = k > 0 ? 1.0f - __builtin_ldexpf(1.0f, -k) : k < -1 ? 1.0f : 0.0f;
    const float B = k >= 0 ? 0.0f : k == -1 ? 0.5f : 1.0f;
    const float y = __builtin_ldexpf(A + (r - e), k) - B;
    const float d = dlk_div_inner(neg ? -y : 2.0f, y + 2.0f);
    const float z = one ? 1.0f : neg ? d : 1.0f - d;
    return __builtin_copysignf(cap * z, x);
}

#endif
