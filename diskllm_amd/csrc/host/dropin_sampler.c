/*
 * dropin_sampler.c -- include/sampler.h on the GPU: the reference's single-row
 * host API (include/sampler.h:19-34, src/sampler.c) as copies around the
 * batched entry points of diskllm_amd.h.
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "diskllm_amd.h"
#include "sampler.h"
#include "dropin.h"

struct sampler {
    sampler_config cfg;
    uint64_t rng;            /* host copy of the xorshift state (src/sampler.c:63) */
    int path;                /* DLK_PATH_* of the first attempt (DLK_DROPIN_PATH, tests) */
    dlk_dropin_ctx dev;
};

sampler *sampler_create(const sampler_config *cfg) {
    if (!cfg) return NULL;
    sampler *s = calloc(1, sizeof(*s));
    if (!s) return NULL;
    s->cfg = *cfg;
    s->rng = dlk_seed_state(cfg->seed);                      /* src/sampler.c:87 */
    /* test hook: the implementation the first attempt of each draw uses (e.g.
     * DLK_PATH_FULL_NO_WAIT to force the sync-timeout recovery below) */
    const char *ps = getenv("DLK_DROPIN_PATH");
    s->path = ps ? atoi(ps) : DLK_PATH_AUTO;
    if (dlk_dropin_init(&s->dev) != 0) {
        free(s);
        return NULL;
    }
    return s;
}

void sampler_free(sampler *s) {
    if (!s) return;
    dlk_dropin_release(&s->dev);
    free(s);
}

/* A device failure the reference API has no channel for: said once on stderr. */
static void report_device_failure(const char *what) {
    static int said;
    if (!said) {
        said = 1;
        fprintf(stderr, "libdiskllm_amd: %s could not reach the GPU; continuing as the reference does "
                        "without its resources (src/sampler.c:145-147)\n", what);
    }
}

/* The reference's greedy_sample (src/sampler.c:9-19) on the host row: the
 * answer of sampler_sample and greedy_sample when the device cannot be reached,
 * as the reference degrades to greedy when it cannot get its work buffer
 * (src/sampler.c:145-147, no random number drawn). */
static int host_greedy(const float *logits, int vocab) {
    int best = 0;
    float bv = logits[0];
    for (int i = 1; i < vocab; i++)
        if (logits[i] > bv) { bv = logits[i]; best = i; }
    return best;
}

/* One row through dlk_sample on `c` with the rng state *rng; on success the
 * token, the status word in *status and the advanced state in *rng_out (not
 * greedy); -1 when a device call fails. */
static int sample_one(dlk_dropin_ctx *c, const float *logits, int vocab, float temperature, int top_k, float top_p,
                      float min_p, int path, const uint64_t *rng, uint64_t *rng_out, uint32_t *status) {
    const size_t row_bytes = (size_t)vocab * sizeof(float);
    if (dlk_dropin_reserve(c, vocab) != 0 || dlk_dropin_reserve_pinned(c, row_bytes + 16) != 0) return -1;
    const int greedy = temperature == 0.0f;
    /* the row through pinned memory in two parts, so that the second is copied
     * on the host while the device takes the first */
    float *pin = (float *)c->pin;
    const int half = vocab / 2 & ~3;
    c->res->rng = *rng;
    if (half > 0) {
        memcpy(pin, logits, (size_t)half * sizeof(float));
        if (dlk_launch_stage_row(c->logits, pin, half, NULL, NULL, NULL, c->stream) != DLK_OK) return -1;
    }
    memcpy(pin + half, logits + half, (size_t)(vocab - half) * sizeof(float));
    if (dlk_launch_stage_row(c->logits + half, pin + half, vocab - half, c->res, c->rng, c->status, c->stream) !=
        DLK_OK)
        return -1;
    dlk_batch b;
    memset(&b, 0, sizeof(b));
    b.logits = c->logits;
    b.ld = vocab;
    b.rng = c->rng;
    b.out_ids = c->ids;
    b.status = c->status;
    dlk_sample_params p;
    memset(&p, 0, sizeof(p));
    p.temperature = temperature;
    p.top_k = top_k;
    p.top_p = top_p;
    p.min_p = min_p;
    p.repeat_penalty = 1.0f;
    p.path = path;
    if (dlk_sample(&b, 1, vocab, &p, c->stream) != DLK_OK) return -1;
    if (dlk_launch_publish_result(c->res, c->rng, c->ids, c->status, c->stream) != DLK_OK) return -1;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return -1;
    *status = c->res->status;
    if (!greedy) *rng_out = c->res->rng;
    return c->res->id;
}

/* The reference always returns a token (src/sampler.c:136-234): its caller
 * feeds it straight to the next decode step (src/cli/main.c:386-388).  A
 * launch whose cross-workgroup wait gave up (another kernel holding the GPU)
 * is run again on the row kernel, which has no such waits, from the same rng
 * state, so the token and the state are the reference's; if the device
 * cannot be reached at all the row is sampled greedily on the host, without
 * drawing, as the reference does when it has no work buffer. */
int sampler_sample(sampler *s, float *logits, int vocab_size) {
    if (!s || !logits || vocab_size <= 0) return -1;
    const sampler_config *cf = &s->cfg;
    uint64_t next = s->rng;
    uint32_t st = 0;
    int id = sample_one(&s->dev, logits, vocab_size, cf->temperature, cf->top_k, cf->top_p, cf->min_p, s->path,
                        &s->rng, &next, &st);
    if (id >= 0 && (st & DLK_STATUS_SYNC_TIMEOUT)) {
        st = 0;
        id = sample_one(&s->dev, logits, vocab_size, cf->temperature, cf->top_k, cf->top_p, cf->min_p, DLK_PATH_ROW,
                        &s->rng, &next, &st);
    }
    if (id < 0 || st != 0 || id >= vocab_size) {
        report_device_failure("sampler_sample");
        return host_greedy(logits, vocab_size);
    }
    if (cf->temperature != 0.0f) s->rng = next;
    return id;
}

int greedy_sample(const float *logits, int vocab_size) {
    if (!logits || vocab_size <= 0) return 0;
    dlk_dropin_ctx *c = dlk_dropin_shared_lock();
    int id = -1;
    uint32_t st = 0;
    if (c) {
        const uint64_t unused = 1;
        uint64_t out = 1;
        id = sample_one(c, logits, vocab_size, 0.0f, 0, 1.0f, 0.0f, DLK_PATH_AUTO, &unused, &out, &st);
        dlk_dropin_shared_unlock();
    }
    if (id < 0 || st != 0 || id >= vocab_size) {
        report_device_failure("greedy_sample");
        return host_greedy(logits, vocab_size);
    }
    return id;
}

/* One penalty op in place on the host row.  Only the touched entries leave the
 * host: the logits of the distinct in-range ids (ids outside [0, vocab) are
 * skipped, as the reference skips them) and their counts go into pinned memory,
 * a kernel applies the op to them there, and the values are written back over
 * those ids: 12 bytes per id over PCIe in place of the whole row.  The order of a
 * history does not matter to either op: repetition scales an entry once per
 * occurrence (its sign never changes), presence subtracts once per distinct id. */
static void report_penalty_failure(uint32_t op) {
    fprintf(stderr, "libdiskllm_amd: sampler_apply_%s_penalty could not reach the GPU; the row was not "
                    "penalised\n", op == DLK_OP_REPETITION ? "repetition" : "presence");
}

static void penalty_one(float *logits, int vocab, const int *seen, int n, uint32_t op, float value) {
    int bits = 6;                                   /* hash slots: at most half of them used */
    while ((size_t)1 << bits < 2 * (size_t)n) bits++;
    const size_t slots = (size_t)1 << bits;
    int32_t *table = calloc(slots, sizeof(int32_t));   /* entry d + 1 of the distinct ids, 0 = free */
    int32_t *ids = malloc((size_t)n * 2 * sizeof(int32_t)), *counts = ids ? ids + n : NULL;
    int done = 0, nd = 0;
    if (table && ids) {
        /* the ids in range, each once, and their counts: before the shared context
         * is taken, so that threads wait for one another's device work alone (and
         * not at all where there is nothing to apply) */
        for (int i = 0; i < n; i++) {
            const int id = seen[i];
            if (id < 0 || id >= vocab) continue;
            /* (the product's high bits: its low ones are those of the id) */
            size_t h = (size_t)(((uint64_t)(uint32_t)id * 0x9E3779B97F4A7C15ull) >> (64 - bits));
            while (table[h] && ids[table[h] - 1] != id) h = (h + 1) & (slots - 1);
            if (table[h]) {
                counts[table[h] - 1]++;
            } else {
                ids[nd] = id;
                counts[nd] = 1;
                table[h] = ++nd;
            }
        }
        done = nd == 0;
    }
    dlk_dropin_ctx *c = nd > 0 ? dlk_dropin_shared_lock() : NULL;
    if (c) {
        if (dlk_dropin_reserve_pinned(c, (size_t)nd * (sizeof(float) + sizeof(int32_t))) == 0) {
            float *vals = (float *)c->pin;
            int32_t *pin_counts = (int32_t *)c->pin + nd;
            for (int d = 0; d < nd; d++) vals[d] = logits[ids[d]];
            memcpy(pin_counts, counts, (size_t)nd * sizeof(int32_t));
            const int ok = dlk_launch_compact_penalty(vals, pin_counts, nd, op, value, c->stream) == DLK_OK;
            if (hipStreamSynchronize(c->stream) == hipSuccess && ok) {
                for (int d = 0; d < nd; d++) logits[ids[d]] = vals[d];
                done = 1;
            }
        }
        dlk_dropin_shared_unlock();
    }
    /* the reference's penalties cannot fail (src/sampler.c:21-52); these can
     * only when host or device memory runs out or the GPU is gone: said on
     * stderr rather than passed over in silence */
    if (!done) report_penalty_failure(op);
    free(table);
    free(ids);
}

void sampler_apply_repetition_penalty(float *logits, int vocab_size, const int *seen_tokens, int num_seen,
                                      float penalty) {
    if (penalty <= 1.0f || !seen_tokens || num_seen <= 0 || !logits || vocab_size <= 0) return;   /* :22 */
    penalty_one(logits, vocab_size, seen_tokens, num_seen, DLK_OP_REPETITION, penalty);
}

void sampler_apply_presence_penalty(float *logits, int vocab_size, const int *seen_tokens, int num_seen,
                                    float presence_penalty) {
    if (presence_penalty == 0.0f || !seen_tokens || num_seen <= 0 || !logits || vocab_size <= 0) return;  /* :36 */
    penalty_one(logits, vocab_size, seen_tokens, num_seen, DLK_OP_PRESENCE, presence_penalty);
}
