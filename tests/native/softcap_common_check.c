/* The branch-free soft-caps (dlk_softcap_common and dlk_softcap_wide on
 * dlk_softcap_quot, compiled for the host) against dlk_softcap_glibc, bit for bit,
 * and the quotient against the IEEE division, over the float bit patterns x = 0,
 * stride, 2 stride, ... of their ranges, for each cap given.  Prints "<checked>
 * <mismatches>" of the common form and of the wide one per cap.  Test
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
        unsigned long long n = 0, bad = 0, wn = 0, wbad = 0;
        for (uint64_t u = 0; recip != 0.0f && u < (1ull << 32); u += stride) {
            const float x = dlk_th_u2f((uint32_t)u), q = dlk_softcap_quot(x, cap, recip);
            if (dlk_softcap_wide_ok(x, q, DLK_SOFTCAP_ONE * cap)) {
                wn++;
                if (dlk_th_f2u(dlk_softcap_wide(x, q, cap, DLK_SOFTCAP_ONE * cap)) != dlk_th_f2u(dlk_softcap_glibc(x, cap)))
                    wbad++;
            }
            if (dlk_softcap_place(q) >= DLK_SOFTCAP_SPAN) continue;
            n++;
            if (q != fabsf(x / cap) || dlk_th_f2u(dlk_softcap_common(x, q, cap)) != dlk_th_f2u(dlk_softcap_glibc(x, cap)))
                bad++;
        }
        printf("%llu %llu %llu %llu\n", n, bad, wn, wbad);
        rc |= bad != 0 || wbad != 0;
    }
    return rc;
}
