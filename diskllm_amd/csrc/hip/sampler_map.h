/*
 * sampler_map.h -- which row and slice of it a workgroup of the fused full-vocabulary
 * kernel takes, and the host's choice among the three mappings.
 *
 * A workgroup waits for the others of its row while it holds its place on the
 * device, so a mapping has to let every row finish when the grid is larger than the
 * device holds.  The device deals workgroups to its N XCDs in turn (b to XCD
 * b % N), and each XCD starts those it is dealt in index order as places come free.
 */
#ifndef DLK_SAMPLER_MAP_H
#define DLK_SAMPLER_MAP_H

#if defined(__HIPCC__)
#define DLK_MAP __host__ __device__ __forceinline__
#else
#define DLK_MAP static inline
#endif

namespace dlk {

enum {
    kMapRows = 0,      /* a row's workgroups consecutive: on each XCD every workgroup of an earlier row
                          comes first, so the first unfinished row never waits for a place behind a
                          later one; on any number of XCDs */
    kMapXcd = 1,       /* each whole group of eight rows interleaved, a row's workgroups eight apart: on
                          eight XCDs a row lies on one (its barriers stay within one L2), where the
                          argument above holds; on fewer, a group of eight rows has to fit the device
                          together */
    kMapHalves = 2     /* a row's workgroups on one XCD of eight, half of them among the first half of
                          that XCD's workgroups, which are the first of their CU, and half among the
                          second, which run behind those (two per CU; older waves win issue): only for
                          a grid that is resident at once, and alone: of two dealt by turns each may
                          hold half of every row.  (64 x 151,936: 42.6 us, 44.0 interleaved) */
};

/* A grid of up to this many workgroups can hold eight places of each XCD, too few
 * (three such beside it) to keep a kMapHalves grid from completing some row. */
constexpr int kMapSmallGrid = 64;

/* `cap`: workgroups that the device holds at once, at least G.  `alone`: no other
 * stream has grids past kMapSmallGrid.  (Interleaved, a grid that waits holds at
 * most G - 1 places of an XCD: four such grids leave one of 64.) */
DLK_MAP int full_map(int rows, int G, int cap, bool alone) {
    if (alone && rows % 8 == 0 && G % 2 == 0 && rows * G <= cap) return kMapHalves;
    return cap >= 8 * G ? kMapXcd : kMapRows;
}

DLK_MAP void full_place(int b, int blocks, int G, int map, int *row, int *g) {
    const int rows8 = (blocks / G) & ~7;           /* rows of whole groups of eight */
    if (map == kMapHalves) {
        /* k: the workgroup's place among its XCD's; each row takes G/2 slices from
         * each half, the first half slice 0 (the start of the draw, the row's longest
         * draw phase) and the last G/2 - 1 (where the top-p crossing of a spread-out
         * row lies, which the others wait for) */
        const int k = b >> 3, R = blocks >> 4, h = G >> 1;
        const int k2 = k < R ? k : k - R, i = k2 % h;
        *row = (k2 / h) * 8 + (b & 7);
        *g = k < R ? (i == 0 ? 0 : G - h + i) : 1 + i;
    } else if (map == kMapXcd && b < rows8 * G) {
        const int k = b >> 3;
        *row = (k / G) * 8 + (b & 7);
        *g = k % G;
    } else {
        *row = b / G;
        *g = b % G;
    }
}

}  // namespace dlk

#endif
