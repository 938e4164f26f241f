/*
 * softcap4.h -- the soft-cap of a group of four logits per lane: the branch-free
 * form of the common range (tanhf_glibc.h) where every lane's four quotients lie in
 * it, the wider branch-free form otherwise, and the general one for the few entries
 * that are outside that too (NaN, quotients between 7.75 and 16 or below 2^-60) and
 * for caps without a safe reciprocal.
 */
#ifndef DLK_SOFTCAP4_H
#define DLK_SOFTCAP4_H

#include "dlk_device.h"
#include "tanhf_glibc.h"

namespace dlk {

DLK_DEV void put4(float (&x)[4], int c, float y) {
    x[0] = c == 0 ? y : x[0];
    x[1] = c == 1 ? y : x[1];
    x[2] = c == 2 ? y : x[2];
    x[3] = c == 3 ? y : x[3];
}

/* x <- cap * tanhf(x / cap); recip from dlk_softcap_recip(cap).  UNROLL: the wide
 * form four times over, for a kernel that has the registers and does nothing else. */
template <bool UNROLL>
DLK_DEV void softcap4(float (&x)[4], float cap, float recip) {
    float q[4];
    uint32_t far = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        q[c] = dlk_softcap_quot(x[c], cap, recip);
        far = max(far, dlk_softcap_place(q[c]));
    }
    if (DLK_HOT(ballot(far >= DLK_SOFTCAP_SPAN) == 0 && recip != 0.0f)) {
#pragma unroll
        for (int c = 0; c < 4; c++) x[c] = dlk_softcap_common(x[c], q[c], cap);
        return;
    }
    const float cap16 = DLK_SOFTCAP_ONE * cap;
    uint32_t odd = 0;                              /* entries left to the general form */
#pragma unroll
    for (int c = 0; c < 4; c++) odd |= recip != 0.0f && dlk_softcap_wide_ok(x[c], q[c], cap16) ? 0u : 1u << c;
    if (recip != 0.0f) {
        if (UNROLL) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float y = dlk_softcap_wide(x[c], q[c], cap, cap16);
                x[c] = (odd >> c) & 1u ? x[c] : y;
            }
        } else {
#pragma unroll 1
            for (int c = 0; c < 4; c++) {
                const float a = c == 0 ? x[0] : c == 1 ? x[1] : c == 2 ? x[2] : x[3];
                const float b = c == 0 ? q[0] : c == 1 ? q[1] : c == 2 ? q[2] : q[3];
                put4(x, c, (odd >> c) & 1u ? a : dlk_softcap_wide(a, b, cap, cap16));
            }
        }
    }
    if (DLK_COLD(ballot(odd != 0) != 0)) {
#pragma unroll 1
        for (int c = 0; c < 4; c++) {
            if (!((odd >> c) & 1u)) continue;
            put4(x, c, dlk_softcap_glibc(c == 0 ? x[0] : c == 1 ? x[1] : c == 2 ? x[2] : x[3], cap));
        }
    }
}

}  // namespace dlk

#endif
