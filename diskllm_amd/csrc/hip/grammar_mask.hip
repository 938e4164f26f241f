/*
 * grammar_mask.hip -- diskllm_grammar_apply_mask (src/core/grammar.c:275-308) for
 * a batch of sequences over one vocabulary.  A token's bytes are read once for
 * all rows: under the JSON validator what a token does to a row depends only on
 * whether the row is inside a string, so one walk of its bytes gives the deepest
 * '}' and ']' it closes for either case, and each row then takes two compares.
 * Rows of the receipt validator are walked from their state through its transition
 * table (grammar_table.h), four states at a time; rows of a block that share a
 * state are walked once.
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

#include "grammar_map.h"
#include "grammar_table.h"

namespace dlk {

constexpr int kMaskBytes = 8192;     /* token bytes staged per block (the rest is read from memory) */

/* How a row tests a token: its string fits (len <= room), closes no more braces
 * and brackets than are open (n, m; as large as can be where nothing is closed),
 * and satisfies the bits below. */
struct __align__(16) RowTest {
    int room;                        /* longest string that still fits the buffer; -1: none */
    int n, m;
    uint32_t bits;
};
constexpr uint32_t kInStr = 1;       /* JSON: inside a string */
constexpr uint32_t kEscaped = 2;     /* JSON: the previous byte is a backslash */
constexpr uint32_t kStart = 4;       /* JSON before its first '{' or '[' */
constexpr uint32_t kFinished = 8;    /* the EOS id's bit */
constexpr uint32_t kWalk = 16;       /* needs the token's walk (JSON) */
constexpr uint32_t kTable = 32;      /* a state of the receipt table */
constexpr uint32_t kScan = 64;       /* any other: resume the row's validator byte by byte */
constexpr int kStateShift = 8;       /* kTable: the state */
constexpr int kFirstShift = 16;      /* kTable: the first row of the block in the same state */

__device__ __forceinline__ RowTest row_test(const dlk_grammar_row &st) {
    RowTest r;
    const dlk_scan_state &s = st.scan;
    /* buffer + string < DLK_GRAMMAR_BUF - 1 (src/core/grammar.c:233) */
    const int64_t room = (int64_t)DLK_GRAMMAR_BUF - 2 - st.bal.len;
    r.room = room < 0 ? -1 : room > 0x7fffffff ? 0x7fffffff : (int)room;
    r.n = r.m = 0x7fffffff;
    r.bits = dlk_balance_finished(&st.bal) ? kFinished : 0u;
    if (!dlk_scan_ok(&s)) {
        r.room = -1;
    } else if (s.mode == DLK_GRAMMAR_JSON && (s.pc == DLK_JS_WS || s.pc == DLK_JS_BODY) && s.n >= 0 && s.m >= 0 &&
               s.flag <= 1) {
        r.n = s.n;
        r.m = s.m;
        r.bits |= kWalk | (s.flag ? kInStr : 0u) | (s.prev == '\\' ? kEscaped : 0u) | (s.pc == DLK_JS_WS ? kStart : 0u);
    } else if (s.mode == DLK_GRAMMAR_JSON || s.mode == DLK_GRAMMAR_RECEIPT) {
        const int key = dlk_receipt_key(&s);
        const uint32_t id = key >= 0 ? kReceiptTable.id[key] : 0u;
        r.bits |= id ? kTable | id << kStateShift : kScan;
    }
    return r;
}

/* Grid (ceil(V / 512), ceil(rows / per)): a block tests its 512 tokens against up
 * to `per` rows.  Bound by latency (offsets, then bytes, then the walk of the
 * block's longest token): the vocabulary is some 1.5 MB.  The token bytes are
 * contiguous, so a block stages them in LDS, eight coalesced loads a thread in
 * flight, and a walk takes four bytes per LDS read.  A walk of dependent byte loads
 * from memory per (token, row) and one atomicAdd per wave and row for the
 * counts (38,000 into one cache line) took 433 us at 16 x 151,936 with counts,
 * this form 15, of which the counting kernel is some 3.  Receipt rows, 16 x
 * 151,936 without counts: 44 us so and 112 when a block resumed its rows' scanner
 * one row after another; 14 now where the rows share a state, 25 where all differ
 * (65 x 1,000: 7.4, 297, 6.6 and 8.7). */
__global__ __launch_bounds__(kMaskTokens) void grammar_mask_kernel(const uint32_t *__restrict__ off,
                                                                   const uint8_t *__restrict__ bytes, int V,
                                                                   const dlk_grammar_row *__restrict__ states,
                                                                   int rows, int per, int eos_id, uint32_t *mask,
                                                                   int64_t mask_ld, float *logits, int64_t ld) {
    __shared__ uint32_t sw[kMaskBytes / 4 + 2];
    __shared__ RowTest tests[kMaskRows];
    __shared__ uint32_t kinds;                     /* the rows' bits, or-ed */
    __shared__ uint64_t words[kMaskRows][kMaskTokens / 64];
    uint8_t *sb = (uint8_t *)sw;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int t0 = blockIdx.x * kMaskTokens, tok = t0 + t;
    const int r0 = blockIdx.y * per, nr = min(per, rows - r0);
    /* (the rows' states first, so that they come while the bytes are staged) */
    dlk_grammar_row st = {};
    if (wave == 0 && lane < nr) st = states[r0 + lane];
    uint32_t b0 = 0, b1 = 0;
    if (tok < V) { b0 = off[tok]; b1 = off[tok + 1]; }
    /* the block's bytes: [lo, lo + n) staged (a token outside is read from memory) */
    const uint32_t lo = off[t0], hi = off[min(t0 + kMaskTokens, V)];
    const int n = hi > lo ? (int)min(hi - lo, (uint32_t)kMaskBytes) : 0;
    for (int i0 = 0; i0 < n; i0 += 8 * kMaskTokens) {
        uint8_t x[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = i0 + k * kMaskTokens + t;
            x[k] = i < n ? bytes[lo + i] : 0;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = i0 + k * kMaskTokens + t;
            if (i < n) sb[i] = x[k];
        }
    }
    if (wave == 0) {
        RowTest r = {};
        if (lane < nr) r = row_test(st);
        if (__ballot((r.bits & kTable) != 0)) {
            const int id = (int)(r.bits & (kTable | 0xffu << kStateShift));
            int first = kMaskRows;
#pragma unroll 1
            for (int i = nr - 1; i >= 0; i--)
                if (id == __builtin_amdgcn_readlane(id, i)) first = i;
            if (r.bits & kTable) r.bits |= (uint32_t)first << kFirstShift;
        }
        if (lane < nr) tests[lane] = r;
        uint32_t any = 0;
        for (uint32_t bit = kWalk; bit <= kScan; bit <<= 1) any |= __ballot((r.bits & bit) != 0) ? bit : 0u;
        if (lane == 0) kinds = any;
    }
    __syncthreads();

    const uint32_t cap = b1 > b0 ? b1 - b0 : 0u;
    const bool staged = cap > 0 && b0 >= lo && b1 <= lo + (uint32_t)n;
    /* bytes i .. i + 3 of the token, 0 past its end */
    auto word_at = [&](uint32_t i) -> uint32_t {
        uint32_t x = 0;
        const uint32_t left = cap - i;
        if (staged) {
            const uint32_t a = b0 - lo + i;
            x = __builtin_amdgcn_alignbyte(sw[(a >> 2) + 1], sw[a >> 2], a & 3u);
            if (left < 4) x &= (1u << (8 * left)) - 1u;
        } else {
            for (uint32_t k = 0; k < 4 && k < left; k++) x |= (uint32_t)bytes[b0 + i + k] << (8 * k);
        }
        return x;
    };
    /* one walk: the string's length (to its first NUL), and for a row outside
     * (0) or inside (1) a string the deepest close of braces and of brackets;
     * quotes toggle, so both cases share one parity */
    int len = 0, lead = 0, par = 0;                /* lead: 0 whitespace so far, 1 then '{' or '[', 2 anything else */
    int db0 = 0, db1 = 0, dk0 = 0, dk1 = 0, nb0 = 0, nb1 = 0, nk0 = 0, nk1 = 0;
    bool quote1 = false, esc = false, ended = false;   /* the first byte is '"'; the last was a backslash */
    const uint32_t any = kinds;
    if (!(any & kWalk)) {
        /* (no JSON row: the string's length is enough) */
        for (uint32_t i = 0; i < cap && !ended; i += 4) {
            const uint32_t x = word_at(i);         /* (bytes past the token's end are 0 too) */
            const uint32_t zero = (x - 0x01010101u) & ~x & 0x80808080u;
            ended = zero != 0;
            len += ended ? __builtin_ctz(zero) >> 3 : 4;
        }
    } else for (uint32_t i = 0; i < cap && !ended; i += 4) {
        const uint32_t x = word_at(i);
        if (i == 0) quote1 = (x & 0xffu) == '"';
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t c = (x >> (8 * k)) & 0xffu;
            ended = ended || c == 0;
            len += ended ? 0 : 1;
            if (lead == 0 && !ended && !dlk_isspace((uint8_t)c)) lead = c == '{' || c == '[' ? 1 : 2;
            const bool quote = c == '"' && !esc && !ended;
            const int s = ended ? 0 : (c == '{') - (c == '}'), d = ended ? 0 : (c == '[') - (c == ']');
            if (par == 0) { db0 += s; nb0 = max(nb0, -db0); dk0 += d; nk0 = max(nk0, -dk0); }
            else { db1 += s; nb1 = max(nb1, -db1); dk1 += d; nk1 = max(nk1, -dk1); }
            par ^= quote ? 1 : 0;
            esc = c == '\\';
        }
    }

    const int fit = len > 0 ? len : 0x7fffffff;    /* the empty string is never allowed (:294-298) */
    const uint32_t flip = quote1 ? kEscaped : 0u;
    uint64_t fed = 0;                              /* bit r: the string passes the validator in row r's state */
    if (any & kTable) {
        /* the block's states four at a time (the same in every thread) */
        for (int r = 0; r < nr;) {
            uint32_t at[4] = {};
            int rows4[4], n4 = 0;
            for (; r < nr && n4 < 4; r++) {
                const uint32_t bits = tests[r].bits;
                if (!(bits & kTable) || (int)(bits >> kFirstShift) != r) continue;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (q == n4) { at[q] = (bits >> kStateShift) & 0xffu; rows4[q] = r; }
                n4++;
            }
            uint32_t x = 0;
            for (int i = 0; i < len && (at[0] | at[1] | at[2] | at[3]); i++) {
                if ((i & 3) == 0) x = word_at((uint32_t)i);
                const uint32_t c = kReceiptTable.cls[x & 0xffu];
#pragma unroll
                for (int q = 0; q < 4; q++) at[q] = kReceiptTable.next[at[q]][c];
                x >>= 8;
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (q < n4 && at[q]) fed |= 1ull << rows4[q];
        }
    }
    if (any & kScan) {
        for (int r = 0; r < nr; r++) {
            if (!(tests[r].bits & kScan)) continue;
            dlk_scan_state s = states[r0 + r].scan;
            uint32_t x = 0;
            for (int i = 0; i < len && dlk_scan_ok(&s); i++) {
                if ((i & 3) == 0) x = word_at((uint32_t)i);
                dlk_scan_step(&s, (uint8_t)x);
                x >>= 8;
            }
            if (dlk_scan_ok(&s)) fed |= 1ull << r;
        }
    }
    auto test_rows = [&](auto validated) {         /* (a loop without `fed` where no row needs it: 16 rows 1 us) */
        for (int r = 0; r < nr; r++) {
            const RowTest R = tests[r];
            /* an escaped first quote does not toggle: the other case's walk from there on */
            const bool in = ((R.bits & kInStr) != 0) != ((R.bits & flip) != 0);
            bool ok = fit <= R.room && len > 0 && R.n >= (in ? nb1 : nb0) && R.m >= (in ? nk1 : nk0) &&
                      !((R.bits & kStart) && lead == 2);
            if (validated && (R.bits & (kTable | kScan)))
                ok = ok && ((fed >> (R.bits & kTable ? R.bits >> kFirstShift : r)) & 1u);
            if (tok == eos_id) ok = (R.bits & kFinished) != 0;           /* :285-291 */
            ok = ok && tok < V;
            const uint64_t bal = __ballot(ok);
            if (lane == 0) words[r][wave] = bal;
        }
    };
    if (any & (kTable | kScan)) test_rows(std::true_type{});
    else test_rows(std::false_type{});
    __syncthreads();
    if (logits && tok < V)
        for (int r = 0; r < nr; r++)
            if (!((words[r][wave] >> lane) & 1u)) logits[(int64_t)(r0 + r) * ld + tok] = -INFINITY;
    const int nw = (V + 31) >> 5, w0 = t0 >> 5;
    const uint32_t *w32 = (const uint32_t *)words;
    for (int i = t; i < nr * (kMaskTokens / 32); i += kMaskTokens) {
        const int r = i / (kMaskTokens / 32), w = i % (kMaskTokens / 32);
        if (w0 + w < nw) mask[(int64_t)(r0 + r) * mask_ld + w0 + w] = w32[i];
    }
}

/* The rows' allowed counts from their finished masks, a block per row; it takes
 * the place of the launch that cleared the counts for atomics. */
__global__ __launch_bounds__(1024) void mask_count_kernel(const uint32_t *__restrict__ mask, int64_t mask_ld, int nw,
                                                          int32_t *valid) {
    __shared__ int part[16];
    const uint32_t *m = mask + (int64_t)blockIdx.x * mask_ld;
    int c = 0;
#pragma unroll 4
    for (int i = threadIdx.x; i < nw; i += 1024) c += __popc(m[i]);
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int i = 0; i < 16; i++) s += part[i];
        valid[blockIdx.x] = s;
    }
}

/* diskllm_grammar_advance (src/core/grammar.c:248-256) as diskllm_sample_grammar
 * calls it after the draw (src/core/sampler_api.c:65-70): unless the token is
 * the EOS id, its string (up to its first NUL) is appended when buffer + string
 * stays below 8191 bytes; here the row's validator and balance states take
 * those bytes.  One thread per row. */
__global__ void grammar_advance_kernel(const uint32_t *__restrict__ off, const uint8_t *__restrict__ bytes, int V,
                                       dlk_grammar_row *states, const int32_t *__restrict__ tokens, int rows,
                                       int eos_id) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    const int tok = tokens[row];
    if (tok < 0 || tok >= V || tok == eos_id) return;
    const uint32_t b0 = off[tok], b1 = off[tok + 1];
    uint32_t len = 0;
    while (b0 + len < b1 && bytes[b0 + len] != 0) len++;
    dlk_grammar_row st = states[row];
    if ((int64_t)st.bal.len + len >= DLK_GRAMMAR_BUF - 1) return;
    for (uint32_t i = 0; i < len; i++) {
        const uint8_t c = bytes[b0 + i];
        dlk_scan_step(&st.scan, c);
        dlk_balance_step(&st.bal, c);
    }
    states[row] = st;
}

}  // namespace dlk

extern "C" int dlk_grammar_mask(const uint32_t *off, const uint8_t *bytes, int vocab, const dlk_grammar_row *states,
                                int rows, int eos_id, uint32_t *mask, int64_t mask_ld, float *logits, int64_t ld,
                                int32_t *valid, hipStream_t stream) {
    using namespace dlk;
    if (!off || !bytes || !states || !mask || vocab <= 0 || rows <= 0 || rows > 65535) return DLK_ERR_INVALID;
    if (mask_ld < (vocab + 31) / 32 || (logits && ld < vocab)) return DLK_ERR_INVALID;
    const int gx = (vocab + kMaskTokens - 1) / kMaskTokens, per = mask_rows_per_block(vocab, rows);
    const int gy = (rows + per - 1) / per;
    hipLaunchKernelGGL(grammar_mask_kernel, dim3(gx, gy), dim3(kMaskTokens), 0, stream, off, bytes, vocab, states, rows,
                       per, eos_id, mask, mask_ld, logits, ld);
    if (valid)
        hipLaunchKernelGGL(mask_count_kernel, dim3(rows), dim3(1024), 0, stream, mask, mask_ld, (vocab + 31) / 32,
                           valid);
    return hipGetLastError() == hipSuccess ? DLK_OK : DLK_ERR_HIP;
}

extern "C" int dlk_grammar_advance(const uint32_t *off, const uint8_t *bytes, int vocab, dlk_grammar_row *states,
                                   const int32_t *tokens, int rows, int eos_id, hipStream_t stream) {
    using namespace dlk;
    if (!off || !bytes || !states || !tokens || vocab <= 0 || rows <= 0) return DLK_ERR_INVALID;
    hipLaunchKernelGGL(grammar_advance_kernel, dim3((rows + 63) / 64), dim3(64), 0, stream, off, bytes, vocab, states,
                       tokens, rows, eos_id);
    return hipGetLastError() == hipSuccess ? DLK_OK : DLK_ERR_HIP;
}

extern "C" int dlk_sample_grammar(const dlk_batch *b, int rows, int vocab, const dlk_sample_params *params,
                                  const uint32_t *off, const uint8_t *bytes, dlk_grammar_row *states, int eos_id,
                                  hipStream_t stream) {
    if (!b || !params || !b->mask || b->mask_row) return DLK_ERR_INVALID;
    /* the batch's mask buffer is written here, then read by the draw */
    int rc = dlk_grammar_mask(off, bytes, vocab, states, rows, eos_id, (uint32_t *)b->mask, b->mask_ld, nullptr, 0,
                              nullptr, stream);
    if (rc != DLK_OK) return rc;
    rc = dlk_sample(b, rows, vocab, params, stream);
    if (rc != DLK_OK) return rc;
    return dlk_grammar_advance(off, bytes, vocab, states, b->out_ids, rows, eos_id, stream);
}
