/* Models the dispatch of the fused kernel's grids (hip/sampler_map.h) on devices of 1 to 8 XCDs and counts the grids
 * in which some row can never finish, for a grid alone and for two that start together past the resident
 * workgroups, and for two to four of any size dealt at random, mapped as grids that share the device are (and, for
 * comparison, in halves).  Also checks that a mapping is one workgroup per slice.  Prints "<grids> <stuck> <pairs>
 * <stuck> <wrong maps> <groups> <stuck> <stuck in halves>".  Test infrastructure. */
#include <stdio.h>
#include <stdlib.h>

#include <utility>
#include <vector>

#include "../../diskllm_amd/csrc/hip/sampler_map.h"

struct Grid {
    int rows, G, map;
    std::vector<int> started, next;    /* workgroups of each row that hold or held a place; each XCD's next one */
};

/* Each XCD has `places`; a row whose workgroups have all started finishes and gives its places back.  burst 0: the
 * grids' workgroups by turns; else at random, up to so many of one grid on one XCD in a row. */
static bool all_finish(std::vector<Grid> grids, int xcds, int places, int burst = 0) {
    std::vector<int> left(xcds, places);
    std::vector<std::vector<std::vector<int>>> held;   /* grid, row -> the XCDs of its places */
    size_t todo = 0, done = 0;
    for (auto &q : grids) {
        held.emplace_back(q.rows);
        todo += q.rows;
        q.started.assign(q.rows, 0);
        q.next.clear();
        for (int x = 0; x < xcds; x++) q.next.push_back(x);
    }
    while (done < todo) {
        bool moved = false;
        auto deal = [&](int x, size_t i) {
            auto &q = grids[i];
            int row, g;
            dlk::full_place(q.next[x], q.rows * q.G, q.G, q.map, &row, &g);
            q.next[x] += xcds;
            left[x]--;
            q.started[row]++;
            held[i][row].push_back(x);
            moved = true;
        };
        auto more = [&](int x, size_t i) { return left[x] > 0 && grids[i].next[x] < grids[i].rows * grids[i].G; };
        if (!burst) {
            for (int x = 0; x < xcds; x++)
                for (size_t n = 0, idle = 0; idle < grids.size(); n++) {
                    const size_t i = n % grids.size();
                    if (more(x, i)) { deal(x, i); idle = 0; }
                    else idle++;
                }
        } else {
            while (true) {
                std::vector<std::pair<int, size_t>> can;
                for (int x = 0; x < xcds; x++)
                    for (size_t i = 0; i < grids.size(); i++)
                        if (more(x, i)) can.push_back({x, i});
                if (can.empty()) break;
                const auto c = can[rand() % can.size()];
                for (int k = 1 + rand() % burst; k > 0 && more(c.first, c.second); k--) deal(c.first, c.second);
            }
        }
        for (size_t i = 0; i < grids.size(); i++)
            for (int r = 0; r < grids[i].rows; r++)
                if (grids[i].started[r] == grids[i].G && !held[i][r].empty()) {
                    for (int x : held[i][r]) left[x]++;
                    held[i][r].clear();
                    done++;
                    moved = true;
                }
        if (!moved) return false;
    }
    return true;
}

int main() {
    long grids = 0, stuck = 0, pairs = 0, stuck2 = 0, wrong = 0;
    for (int xcds = 1; xcds <= 8; xcds *= 2)
        for (int places : {32, 64})
            for (int G = 1; G <= 16; G++)
                for (int rows : {1, 5, 7, 8, 9, 16, 23, 24, 31, 40, 64, 67, 96, 129, 256, 300}) {
                    const int cap = xcds * places;
                    if (cap < G) continue;
                    const Grid q{rows, G, dlk::full_map(rows, G, cap, true), {}, {}};
                    std::vector<char> seen(rows * G, 0);
                    for (int b = 0; b < rows * G; b++) {
                        int row = -1, g = -1;
                        dlk::full_place(b, rows * G, G, q.map, &row, &g);
                        if (row < 0 || row >= rows || g < 0 || g >= G || seen[row * G + g]++) wrong++;
                    }
                    grids++;
                    if (!all_finish({q}, xcds, places)) stuck++;
                    if (rows * G > cap && places == 64 && xcds == 8) {
                        const Grid other{rows / 2 + 33, 16, dlk::full_map(rows / 2 + 33, 16, cap, true), {}, {}};
                        pairs++;
                        if ((rows / 2 + 33) * 16 > cap && !all_finish({q, other}, xcds, places)) stuck2++;
                    }
                }
    long groups = 0, stuck3 = 0, halves = 0;
    srand(11);
    for (int n = 2; n <= 4; n++)
        for (int burst : {1, 8, 64})
            for (int it = 0; it < 150; it++) {
                std::vector<Grid> q, h;
                for (int i = 0; i < n; i++) {
                    const int G = 2 + 2 * (rand() % 8), rows = rand() % 3 ? 8 * (1 + rand() % 40) : 1 + rand() % 300;
                    q.push_back({rows, G, dlk::full_map(rows, G, 512, false), {}, {}});
                    h.push_back({64, 8, dlk::full_map(64, 8, 512, true), {}, {}});
                }
                groups++;
                if (!all_finish(q, 8, 64, burst)) stuck3++;
                if (!all_finish(h, 8, 64, burst)) halves++;
            }
    printf("%ld %ld %ld %ld %ld %ld %ld %ld\n", grids, stuck, pairs, stuck2, wrong, groups, stuck3, halves);
    return 0;
}
