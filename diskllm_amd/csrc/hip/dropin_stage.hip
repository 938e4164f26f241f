/*
 * dropin_stage.hip -- the host-pointer drop-ins' traffic between pinned host
 * memory and the device, as kernels of the call's own stream.
 *
 * A drop-in call is one row and waits for its answer, so what counts is latency:
 * copies by the DMA engines wait for a signal between queues at each end (three
 * small results copied back one by one, and a pageable row up, made sampler_sample
 * 105 us around a 31 us kernel).  The host writes the row into pinned memory, a
 * kernel takes it over PCIe and stays in order with the sampling kernels behind
 * it, and one lane writes the results back.
 */
#include <hip/hip_runtime.h>

#include "../../../include/diskllm_amd.h"
#include "../host/dropin.h"
#include "dlk_device.h"

namespace dlk {

constexpr int kStageThreads = 256;
constexpr int kStagePer = 4;          /* 16-byte loads in flight per thread: 608 KB are 38 blocks' worth at once */

/* dst[0 .. n4) <- src (pinned host memory), four floats at a time; the call's
 * rng state and a clear status word with it */
__global__ __launch_bounds__(kStageThreads) void stage_row_kernel(float4 *__restrict__ dst,
                                                                  const float4 *__restrict__ src, int n4,
                                                                  const dlk_dropin_result *res, uint64_t *rng,
                                                                  uint32_t *status) {
    const int i0 = blockIdx.x * kStageThreads * kStagePer + threadIdx.x;
    float4 x[kStagePer];
#pragma unroll
    for (int k = 0; k < kStagePer; k++)
        if (i0 + k * kStageThreads < n4) x[k] = src[i0 + k * kStageThreads];
#pragma unroll
    for (int k = 0; k < kStagePer; k++)
        if (i0 + k * kStageThreads < n4) dst[i0 + k * kStageThreads] = x[k];
    if (res && i0 == 0) {
        *rng = res->rng;
        *status = 0u;
    }
}

__global__ void publish_result_kernel(dlk_dropin_result *res, const uint64_t *rng, const int32_t *id,
                                      const uint32_t *status) {
    res->rng = *rng;
    res->id = *id;
    res->status = *status;
}

}  // namespace dlk

extern "C" int dlk_launch_stage_row(float *dst, const float *src, int n, const dlk_dropin_result *res, uint64_t *rng,
                                    uint32_t *status, hipStream_t stream) {
    using namespace dlk;
    const int n4 = (n + 3) / 4, per = kStageThreads * kStagePer;
    hipLaunchKernelGGL(stage_row_kernel, dim3((n4 + per - 1) / per), dim3(kStageThreads), 0, stream, (float4 *)dst,
                       (const float4 *)src, n4, res, rng, status);
    return hipGetLastError() == hipSuccess ? DLK_OK : DLK_ERR_HIP;
}

extern "C" int dlk_launch_publish_result(dlk_dropin_result *res, const uint64_t *rng, const int32_t *id,
                                         const uint32_t *status, hipStream_t stream) {
    hipLaunchKernelGGL(dlk::publish_result_kernel, dim3(1), dim3(1), 0, stream, res, rng, id, status);
    return hipGetLastError() == hipSuccess ? DLK_OK : DLK_ERR_HIP;
}
