/*
 * softcap.hip -- the reference's logit soft-cap on the device, in place:
 * logits[i] = cap * tanhf(logits[i] / cap) over each row
 * (src/core/context.c:604-606 after a prefill, :873-876 after a decode step,
 * where it is a host loop over the vocabulary).  tanhf is bit-identical to the
 * host libm's (tanhf_glibc.h).
 *
 * Elementwise work of 8 bytes per element (read + write) that the general form's
 * 80 vector instructions per element and its branches made VALU-bound: at
 * 512 x 262,144 320 to 540 us over fresh logits, by how wide they lie (a copy of that
 * size takes 208).  A group of four whose quotients lie in the common range in every
 * lane takes the branch-free form of some 60 instructions, other groups the wide one
 * of some 75 (softcap4.h): 189 us at cap 30 and sd 4, 211 at sd 5, 222 to 229 at sd
 * 10 and 30 and at cap 15 and sd 5 (415, 561 and 417 while one value past the common
 * range sent its group to the general form).  Rows of any alignment take 16-byte
 * loads and stores (4-byte alignment is enough); a workgroup covers
 * 4 * 256 * kSoftcapVec4 elements of one row.
 */
#include <hip/hip_runtime.h>

#include "softcap4.h"
#include "../../../include/diskllm_amd.h"

namespace dlk {

constexpr int kSoftcapThreads = 256;
constexpr int kSoftcapVec4 = 1;             /* groups of four per thread (2: 216 us, 4: 221 at 512 x 262,144) */

__global__ __launch_bounds__(kSoftcapThreads) void softcap_vec_kernel(float *__restrict__ logits, int64_t ld,
                                                                      int vocab, float cap, float recip) {
    float *row = logits + (int64_t)blockIdx.y * ld;
    const int base = (blockIdx.x * kSoftcapVec4 * kSoftcapThreads + threadIdx.x) * 4;
    float4 v[kSoftcapVec4];
#pragma unroll
    for (int k = 0; k < kSoftcapVec4; k++) {
        const int i = base + k * kSoftcapThreads * 4;
        if (i + 3 < vocab) v[k] = load4(row + i);
    }
#pragma unroll
    for (int k = 0; k < kSoftcapVec4; k++) {
        const int i = base + k * kSoftcapThreads * 4;
        if (i + 3 < vocab) {
            float x[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
            softcap4<true>(x, cap, recip);
            store4(row + i, make_float4(x[0], x[1], x[2], x[3]));
        } else {
            for (int c = 0; c < 4 && i + c < vocab; c++) row[i + c] = dlk_softcap_glibc(row[i + c], cap);
        }
    }
}

}  // namespace dlk

extern "C" int dlk_softcap(float *logits, int64_t ld, int rows, int vocab, float cap, hipStream_t stream) {
    if (!logits || rows < 0 || vocab < 0 || ld < vocab) return DLK_ERR_INVALID;
    if (rows > 65535 || vocab > 0x7fffffff - 8192) return DLK_ERR_UNSUPPORTED;   /* grid rows; int indices */
    /* the reference caps only when the model's cap is positive (a NaN cap too is no cap) */
    if (rows == 0 || vocab == 0 || !(cap > 0.0f)) return DLK_OK;
    const int per = 4 * dlk::kSoftcapVec4 * dlk::kSoftcapThreads;
    const dim3 grid((unsigned)((vocab + per - 1) / per), (unsigned)rows);
    hipLaunchKernelGGL(dlk::softcap_vec_kernel, grid, dim3(dlk::kSoftcapThreads), 0, stream, logits, ld, vocab, cap,
                       dlk_softcap_recip(cap));
    return hipGetLastError() == hipSuccess ? DLK_OK : DLK_ERR_HIP;
}
