/* The branch-free soft-cap (dlk_softcap_common on dlk_softcap_quot, compiled for
 * the host) against dlk_softcap_glibc, bit for bit, and its quotient against the
 * IEEE division, over the float bit patterns x = 0, stride, 2 stride, ... of its
 * range, for each cap given.  Prints "<checked> <mismatches>" per cap.  Test
 * infrastructure. */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include "../../diskllm_amd/csrc/hip/tanhf_glibc.h"

int main(int argc, char **argv) {
    const uint64_t stride = strtoull(argv[1], 0, 0);
    int rc = 0;
    for (int a = 2; a < argc; a++) {
        const float cap = strtof(argv[a], NULL), recip = dlk_softcap_recip(cap);
        unsigned long long n = 0, bad = 0;
        for (uint64_t u = 0; recip != 0.0f && u < (1ull << 32); u += stride) {
            const float x = dlk_th_u2f((uint32_t)u), q = dlk_softcap_quot(x, cap, recip);
            if (dlk_softcap_place(q) >= DLK_SOFTCAP_SPAN) continue;
            n++;
            if (q != fabsf(x / cap) || dlk_th_f2u(dlk_softcap_common(x, q, cap)) != dlk_th_f2u(dlk_softcap_glibc(x, cap)))
                bad++;
        }
        printf("%llu %llu\n", n, bad);
        rc |= bad != 0;
    }
    return rc;
}
