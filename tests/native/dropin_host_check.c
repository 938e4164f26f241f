/* The drop-in penalty calls (host/dropin_sampler.c, host/dropin_ctx.c) on stand-ins for the HIP runtime: what they do
 * on the host around the one kernel.  Prints "ok" or the line that failed.  Test infrastructure. */
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

#include "../../include/diskllm_amd.h"
#include "../../include/sampler.h"
#include "../../diskllm_amd/csrc/host/dropin.h"

static int g_calls, g_fail, g_launched;            /* runtime calls; make them fail; ids in the last launch */

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; g_calls++; *s = (hipStream_t)1; return g_fail ? hipErrorNoDevice : hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; g_calls++; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { g_calls++; *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; g_calls++; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
int dlk_release_stream(hipStream_t s) { (void)s; return DLK_OK; }
int dlk_sample(const dlk_batch *b, int rows, int vocab, const dlk_sample_params *p, hipStream_t s) { (void)b; (void)rows; (void)vocab; (void)p; (void)s; return DLK_ERR_HIP; }
uint64_t dlk_seed_state(uint64_t s) { return s; }
int dlk_launch_stage_row(float *d, const float *s, int n, const dlk_dropin_result *r, uint64_t *g, uint32_t *st, hipStream_t q) { (void)d; (void)s; (void)n; (void)r; (void)g; (void)st; (void)q; return DLK_OK; }
int dlk_launch_publish_result(dlk_dropin_result *r, const uint64_t *g, const int32_t *i, const uint32_t *st, hipStream_t q) { (void)r; (void)g; (void)i; (void)st; (void)q; return DLK_OK; }
int dlk_launch_compact_penalty(float *v, const int32_t *counts, int n, uint32_t op, float value, hipStream_t s) {
    (void)s;
    g_launched = n;
    for (int i = 0; i < n; i++)
        for (int c = 0; c < (op == DLK_OP_REPETITION ? counts[i] : 1); c++)
            v[i] = op == DLK_OP_PRESENCE ? v[i] - value : v[i] < 0 ? v[i] * value : v[i] / value;
    return DLK_OK;
}

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

enum { V = 262144, N = 8192 };
static float row[V], want[V];
static int outside[4] = {-1, V, V + 7, -2147483647};
static volatile int done;

static void *call(void *a) {
    (void)a;
    sampler_apply_presence_penalty(row, V, outside, 4, 0.5f);
    done = 1;
    return NULL;
}

int main(int argc, char **argv) {
    /* ids that are all out of range: nothing to apply, whether there is a device or not */
    g_fail = argc > 1 && strcmp(argv[1], "nodevice") == 0;
    sampler_apply_repetition_penalty(row, V, outside, 4, 1.5f);
    sampler_apply_presence_penalty(row, V, outside, 4, 0.5f);
    CHECK(g_calls == 0);
    if (g_fail) { printf("ok\n"); return 0; }
    /* and no waiting for another thread's call */
    CHECK(dlk_dropin_shared_lock() != NULL);
    pthread_t th;
    pthread_create(&th, NULL, call, NULL);
    for (int i = 0; i < 200 && !done; i++) nanosleep(&(struct timespec){0, 10000000}, NULL);
    const int early = done;
    dlk_dropin_shared_unlock();
    pthread_join(th, NULL);
    CHECK(early);
    /* ids with repeats, some outside, some whose hashes lie close: each counted once */
    static int seen[N];
    for (int kind = 0; kind < 4; kind++) {
        int in = 0, distinct = 0;
        static int count[V];
        memset(count, 0, sizeof count);
        for (int i = 0; i < N; i++) {
            seen[i] = kind == 0 ? (i * 32) % V : kind == 1 ? (i % 256) << 10 : kind == 2 ? i % 7 - 3 : (int)((i * 2654435761u) % (V + 50)) - 20;
            if (seen[i] >= 0 && seen[i] < V) { in++; distinct += count[seen[i]]++ == 0; }
        }
        for (int i = 0; i < V; i++) {
            row[i] = (float)(i % 13) - 6.0f;
            want[i] = row[i];
            for (int c = 0; c < count[i]; c++) want[i] = want[i] < 0 ? want[i] * 1.25f : want[i] / 1.25f;
        }
        sampler_apply_repetition_penalty(row, V, seen, N, 1.25f);
        CHECK(in > 0 && g_launched == distinct);
        CHECK(memcmp(row, want, sizeof row) == 0);
    }
    printf("ok\n");
    return 0;
}
