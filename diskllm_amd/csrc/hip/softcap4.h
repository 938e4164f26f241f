/*
 * softcap4.h -- the soft-cap of a group of four logits per lane: the branch-free
 * form (tanhf_glibc.h) where every lane's four quotients lie in its range, the
 * general one otherwise (one rolled copy, out of the main path).
 */
#ifndef DLK_SOFTCAP4_H
#define DLK_SOFTCAP4_H

#include "dlk_device.h"
#include "tanhf_glibc.h"

namespace dlk {

/* x <- cap * tanhf(x / cap); recip from dlk_softcap_recip(cap) */
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
    } else {
#pragma unroll 1
        for (int c = 0; c < 4; c++) {
            const float y = dlk_softcap_glibc(c == 0 ? x[0] : c == 1 ? x[1] : c == 2 ? x[2] : x[3], cap);
            x[0] = c == 0 ? y : x[0];
            x[1] = c == 1 ? y : x[1];
            x[2] = c == 2 ? y : x[2];
            x[3] = c == 3 ? y : x[3];
        }
    }
}

}  // namespace dlk

#endif
