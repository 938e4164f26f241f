/*
 * grammar_map.h -- how many tokens and rows a block of the grammar mask kernel takes.
 */
#ifndef DLK_GRAMMAR_MAP_H
#define DLK_GRAMMAR_MAP_H

#include <algorithm>

namespace dlk {

constexpr int kMaskTokens = 512;     /* a thread per token: 16 mask words, one 64-byte line per row and block */
constexpr int kMaskRows = 64;        /* rows per block at most (a wave's lanes, a word's bits) */
constexpr int kMaskCus = 256;
constexpr int kMaskBlocks = 300;

/* Rows are split over blocks as long as each block has a CU to itself: a JSON row
 * costs its block some 0.2 us, a second block on a CU some 2 (2 x 75,392: 8.9 us in 148
 * blocks, 11.2 in 296).  Past that the split goes on, up to about kMaskBlocks blocks,
 * while each keeps 16 rows: 16 x 32,000 9.2 us (11.4 in 63 blocks of 16 rows), 64 x
 * 32,000 11.4 (20.6 in 63 of 64, 13.3 in 315), 64 x 50,257 14.4 (20.9 in 99 of 64),
 * 64 x 151,936 22.1 (26.4 in 297 of 64). */
static inline int mask_rows_per_block(int vocab, int rows) {
    const int gx = (vocab + kMaskTokens - 1) / kMaskTokens;
    const int alone = std::min(rows, kMaskCus / gx);
    const int wide = std::min(rows / 16, (kMaskBlocks + gx - 1) / gx);
    const int gy = std::max({(rows + kMaskRows - 1) / kMaskRows, alone, wide});
    return (rows + gy - 1) / gy;
}

} /* namespace dlk */

#endif
