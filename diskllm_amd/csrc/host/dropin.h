/*
 * dropin.h -- device staging shared by the host-pointer drop-ins (sampler.h,
 * grammar.h): one stream and grow-only device buffers per context.
 */
#ifndef DLK_DROPIN_H
#define DLK_DROPIN_H

#include <stdint.h>

#include <hip/hip_runtime_api.h>

/* What a sampling call sends up and brings back beside the row (pinned). */
typedef struct {
    uint64_t rng;
    int32_t id;
    uint32_t status;
} dlk_dropin_result;

typedef struct {
    hipStream_t stream;
    float *logits;       /* [cap] */
    int cap;             /* a multiple of 4 */
    dlk_dropin_result *res;   /* pinned host memory */
    unsigned char *pin;  /* pinned host memory: the row going up, or a penalty's values and counts */
    size_t pin_cap;
    uint64_t *rng;       /* [1] */
    int32_t *ids;        /* [2]: token, valid count */
    uint32_t *status;    /* [1] */
    uint32_t *mask;      /* [mask_cap] words */
    int mask_cap;
} dlk_dropin_ctx;

int dlk_dropin_init(dlk_dropin_ctx *c);
void dlk_dropin_release(dlk_dropin_ctx *c);
int dlk_dropin_reserve(dlk_dropin_ctx *c, int vocab);
/* At least `bytes` of pinned staging (16-byte aligned; contents lost when it grows). */
int dlk_dropin_reserve_pinned(dlk_dropin_ctx *c, size_t bytes);

#ifdef __cplusplus
extern "C" {
#endif
/* dst[0 .. n) <- pinned src, rounded up to whole groups of four; with res, its rng
 * state to *rng and a clear *status (hip/dropin_stage.hip). */
int dlk_launch_stage_row(float *dst, const float *src, int n, const dlk_dropin_result *res, uint64_t *rng,
                         uint32_t *status, hipStream_t stream);
int dlk_launch_publish_result(dlk_dropin_result *res, const uint64_t *rng, const int32_t *id, const uint32_t *status,
                              hipStream_t stream);
/* One penalty op in place on n compact pinned values with their ids' counts (hip/penalties.hip). */
int dlk_launch_compact_penalty(float *vals, const int32_t *counts, int n, uint32_t op, float value,
                               hipStream_t stream);
#ifdef __cplusplus
}
#endif

/* The process-wide context of the stateless calls, locked while in use. */
dlk_dropin_ctx *dlk_dropin_shared_lock(void);
void dlk_dropin_shared_unlock(void);

#endif
