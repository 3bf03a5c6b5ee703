// Host-side check of a flat launch's split (leap::flat_segment and the
// records around it): for random item lengths, workgroup counts and start
// costs, the segments of all workgroups cover every item's rows once, number
// its chunks 0..n_local-1 in the order of their rows, and use records of
// their own inside the launch's, chunk records consecutive per item and
// sub-group records apart.  Built and run by tests/test_flat_split.py.
#include "decode_attention.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <vector>
#define REQUIRE(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
int main() {
    std::mt19937 rng(1);
    auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    long long n_segments = 0;
    for (int trial = 0; trial < 20000; trial++) {
        const int n_wg = (int[]){1, 8, 32, 64}[rng() % 4], n_items = pick(1, leap::kFlatMaxItems);
        const int longest = (int[]){1, 5, 64, 300, 9000, 131072}[rng() % 6], start = (int[]){0, 1, leap::kFlatSegmentRows}[rng() % 3];
        const bool equal = rng() % 4 == 0;
        std::vector<int> T(n_items), end(n_items);
        int total = 0;
        for (int i = 0; i < n_items; i++) {
            T[i] = equal ? longest : rng() % 8 == 0 ? 0 : pick(1, longest);  // 0: a position the launch cannot serve
            total += T[i] ? T[i] + start : 0;
            end[i] = total;
        }
        const int run = std::max((total + n_wg - 1) / n_wg, leap::kFlatMinRun);
        std::vector<int> rows(n_items, 0), chunks(n_items, 0), n_local(n_items, 0), first_rec(n_items, -1);
        std::map<int, int> rec_of, sub_of;
        for (int w = 0; w < n_wg; w++) {
            int at = w * run;
            const int stop = std::min(at + run, total);
            while (at < stop) {
                int i = 0;
                while (end[i] <= at) i++;
                const leap::FlatSegment f = leap::flat_segment(w, run, at, stop, i, end[i] - (T[i] + start), end[i], start);
                at = end[i];
                if (f.begin == f.end) continue;
                n_segments++;
                REQUIRE(f.item == i && f.pos == T[i] - 1);
                REQUIRE(f.begin == rows[i] && f.end > f.begin && f.end <= T[i]);
                rows[i] = f.end;
                REQUIRE(f.lc == chunks[i] && f.lc < f.n_local && f.n_local <= n_wg);
                chunks[i]++;
                n_local[i] = f.n_local;
                if (f.lc == 0) first_rec[i] = f.rec0;
                REQUIRE(f.rec0 == first_rec[i]);
                REQUIRE(f.rec0 + f.lc < n_wg + n_items && rec_of.emplace(f.rec0 + f.lc, i).second);
                const int sub = leap::flat_sub_record(n_wg, n_items, f.rec0, i) + f.lc / leap::kSubGroup;
                REQUIRE(sub >= n_wg + n_items && sub < leap::flat_records(n_wg, n_items));
                const int owner = i * 1000 + f.lc / leap::kSubGroup;
                REQUIRE(sub_of.emplace(sub, owner).first->second == owner);
            }
        }
        for (int i = 0; i < n_items; i++) REQUIRE(rows[i] == T[i] && chunks[i] == (T[i] ? n_local[i] : 0));
    }
    std::printf("segments %lld ok\n", n_segments);
}
