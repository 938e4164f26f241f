/* The host side of dlk_sample (hip/capi.hip, compiled for the host alone) on stand-ins for the HIP runtime and the
 * kernel launches, so that what it does around them can be looked at without a device: which calls it makes, in
 * which order and on which stream, and what it does when memory runs out or a stream is being captured.  Memory
 * addresses are made up and never read.  Prints one line per call of interest.  Test infrastructure. */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include <hip/hip_runtime_api.h>

#include "../../include/diskllm_amd.h"
#include "../../diskllm_amd/csrc/hip/sampler_params.h"
#include "../../diskllm_amd/csrc/hip/sampler_full.h"
#include "../../diskllm_amd/csrc/hip/sampler_topk.h"

static size_t g_memory = (size_t)1 << 40;          /* what hipMalloc can give in one piece */
static int g_resident = 512;                       /* workgroups of the fused kernel resident at once */
static hipStreamCaptureStatus g_capture = hipStreamCaptureStatusNone;
static hipError_t g_last = hipSuccess;             /* as the runtime keeps it until it is asked for */
static std::map<const void *, std::string> g_kernels;
static std::map<void *, size_t> g_blocks;
static char *g_next = (char *)0x100000000ull;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (g_capture != hipStreamCaptureStatusNone) { printf("malloc under capture\n"); return g_last = hipErrorStreamCaptureUnsupported; }
    if (n > g_memory) { printf("malloc failed\n"); return g_last = hipErrorOutOfMemory; }
    *p = g_next;
    g_next += (n + 0xffffff) & ~(size_t)0xffffff;
    g_blocks[*p] = n;
    printf("malloc %zu\n", n);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (p) printf("free %s\n", g_blocks.erase(p) ? "block" : "UNKNOWN");
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { printf("memset on the null stream\n"); return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = (void *)0x80000000ull; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { *s = g_capture; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { printf("synchronize stream %zu\n", (size_t)s); return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t s) {
    const std::string &n = g_kernels[f];
    printf("%s on stream %zu\n", n.find("zero_words") != std::string::npos ? "clear" : n.c_str(), (size_t)s);
    return g_last;
}
static struct { dim3 g, b; size_t lds; hipStream_t s; } g_cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { g_cfg = {g, b, lds, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = g_cfg.g; *b = g_cfg.b; *lds = g_cfg.lds; *s = g_cfg.s;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) { g_kernels[f] = name; }
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}

static int launched(void) { return hipGetLastError() == hipSuccess ? 0 : -1; }
int dlk_launch_row_kernel(const dlk::RowParams *, int rows, size_t, hipStream_t s) { printf("row kernel, %d rows on stream %zu\n", rows, (size_t)s); return launched(); }
int dlk_launch_topk_kernel(const dlk::TopkParams *f, int rows, size_t, hipStream_t s) {
    printf("top-k kernel, %d rows on stream %zu\n", rows, (size_t)s);
    printf("slices %d\n", f->G);
    return launched();
}
int dlk_topk_kernel_occupancy(int, size_t) { return 8; }
int dlk_launch_full_kernel(const dlk::FullParams *f, int rows, int, size_t, hipStream_t s) {
    printf("fused kernel, %d rows on stream %zu\n", rows, (size_t)s);
    printf("mapping %d\n", f->map);
    return launched();
}
int dlk_full_kernel_capacity(int, size_t, int, int) { return g_resident; }
int dlk_launch_long_history_penalties(float *, int64_t, int, int, const int32_t *, const int32_t *, uint32_t, float, float, float, int, int32_t *, const uint64_t *, uint64_t *, hipStream_t) { printf("penalties\n"); return launched(); }
int dlk_launch_long_history_fixup(int, const int32_t *, const uint64_t *, uint64_t *, int32_t *, uint32_t *, hipStream_t) { return launched(); }
int dlk_launch_prepare_rows(const float *, int64_t, float *, int64_t, int, int, const uint32_t *, int64_t, const int32_t *, float, hipStream_t) { printf("prepare\n"); return launched(); }
}

/* commands: "memory N", "resident N", "capture 0|1", "release S", "history N" (longest history of the next calls),
 * "sample ROWS VOCAB LD TOPK TEMPERATURE STREAM" */
int main(int argc, char **argv) {
    int history = 0;
    for (int i = 1; i < argc;) {
        const std::string c = argv[i++];
        if (c == "memory") g_memory = strtoull(argv[i++], 0, 0);
        else if (c == "resident") g_resident = atoi(argv[i++]);
        else if (c == "capture") g_capture = atoi(argv[i++]) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
        else if (c == "history") history = atoi(argv[i++]);
        else if (c == "release") printf("release %d\n", dlk_release_stream((hipStream_t)strtoull(argv[i++], 0, 0)));
        else {
            dlk_batch b;
            dlk_sample_params p;
            memset(&b, 0, sizeof b);
            memset(&p, 0, sizeof p);
            const int rows = atoi(argv[i]), vocab = atoi(argv[i + 1]);
            b.logits = (const float *)0x10000000ull;
            b.out_ids = (int32_t *)0x20000000ull;
            b.rng = (uint64_t *)0x30000000ull;
            b.ld = atoll(argv[i + 2]);
            p.top_k = atoi(argv[i + 3]);
            p.temperature = strtof(argv[i + 4], 0);
            p.top_p = 0.9f;
            p.repeat_penalty = 1.0f;
            if (history) {
                b.hist_off = b.hist_ids = (const int32_t *)0x40000000ull;
                p.max_history = history;
            }
            const hipStream_t s = (hipStream_t)strtoull(argv[i + 5], 0, 0);
            i += 6;
            printf("status %d\n", dlk_sample(&b, rows, vocab, &p, s));
        }
    }
    return 0;
}
