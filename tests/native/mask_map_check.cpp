/* How the grammar mask kernel splits rows over blocks (hip/grammar_map.h): prints "<shapes> <wrong> <crowded>", crowded
 * being the shapes whose blocks share CUs for fewer than 16 rows each.  Test infrastructure. */
#include <stdio.h>

#include "../../diskllm_amd/csrc/hip/grammar_map.h"

int main() {
    long shapes = 0, wrong = 0, crowded = 0;
    for (int vocab = 1; vocab < 600000; vocab += vocab < 1200 ? 1 : 997)
        for (int rows = 1; rows <= 65535; rows += rows < 600 ? 1 : 4639) {
            const int gx = (vocab + dlk::kMaskTokens - 1) / dlk::kMaskTokens, per = dlk::mask_rows_per_block(vocab, rows);
            shapes++;
            if (per < 1 || per > dlk::kMaskRows) { wrong++; continue; }
            const int gy = (rows + per - 1) / per, least = (rows + dlk::kMaskRows - 1) / dlk::kMaskRows;
            if (gx * gy > dlk::kMaskCus && gy > least && per < 16) crowded++;
        }
    printf("%ld %ld %ld\n", shapes, wrong, crowded);
    return 0;
}
