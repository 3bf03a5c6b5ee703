// Host-side check of the rules that size and route a launch, on the library's
// own source (no device): over every supported head shape, handles of 1-128
// sequences, fewer sequences than the handle holds, and row counts given or
// estimated, a flat launch's kernel exists and its records and counters fit
// in the handle's workspace.  Built and run by tests/test_launch_rules.py.
#include "checkpoint.cpp"
#include "leap_hip_attention.hip"

#include <cstdlib>
#include <set>

#define REQUIRE(c, ...)                                      \
    do {                                                     \
        if (!(c)) {                                          \
            std::printf("line %d: %s: ", __LINE__, #c);      \
            std::printf(__VA_ARGS__);                        \
            std::printf("\n");                               \
            std::exit(1);                                    \
        }                                                    \
    } while (0)

int main()
{
    long long calls = 0, flat = 0, flat_partial = 0, split_views = 0;
    for (int n_cu : {256, 128, 64, 32})
        for (int hd : {64, 128})
            for (int g : {1, 2, 3, 4, 8, 16})
                for (int nkv : {1, 2, 3, 4, 5, 8, 10, 16, 32, 40})
                    for (int max_batch : {1, 2, 3, 4, 5, 8, 16, 33, 64, 128}) {
                        leap_hip_attention_config c{};
                        c.n_layers = c.layer_end = 1;
                        c.n_heads = g * nkv;
                        c.n_kv_heads = nkv;
                        c.head_dim = hd;
                        c.seq_len = 32768;
                        c.max_batch = max_batch;
                        const Workspace w = workspace_for(c, n_cu);
                        leap_hip_attention h;
                        h.cfg = c;
                        h.group = g;
                        h.n_cu = n_cu;
                        h.max_chunks = w.max_chunks;
                        h.max_flat = w.max_flat;
                        std::set<int> ns;
                        for (int n : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64, 100, 128}) ns.insert(std::min(n, max_batch));
                        for (int n_seq : ns)
                            for (int max_T : {1, 31, 64, 100, 500, 1000, 1024, 2011, 3000, 4095, 4096, 5000, 6143, 8192,
                                              12288, 16384, 24576, 32768})
                                // estimated (total_rows 0), equal lengths, ragged ones, one long among short
                                for (long long rows : {(long long)n_seq * max_T / 2 + 1, (long long)n_seq * max_T,
                                                       (long long)n_seq * max_T * 5 / 6, (long long)max_T + n_seq - 1}) {
                                    calls++;
                                    const LaunchShape s = launch_view(shape_of(&h), n_seq, rows);
                                    if (s.kv_split != shape_of(&h).kv_split) split_views++;
                                    const int n_wg = flat_launch(s, n_seq, rows, max_T);
                                    if (!n_wg) continue;
                                    flat++;
                                    flat_partial += n_seq < max_batch;
                                    char what[160];
                                    std::snprintf(what, sizeof what, "%d CUs, heads %d/%d/%d, %d of %d sequences, longest %d, rows %lld",
                                                  n_cu, c.n_heads, nkv, hd, n_seq, max_batch, max_T, rows);
                                    REQUIRE((hd == 64 ? pick_flat<64>(s.group, s.kv_split) : pick_flat<128>(s.group, s.kv_split)),
                                            "%s", what);
                                    const int groups = n_seq * s.n_kv_heads, items = (groups + leap::kXcds - 1) / leap::kXcds;
                                    REQUIRE(items <= leap::kFlatMaxItems, "%s", what);
                                    REQUIRE((size_t)leap::kXcds * s.group * leap::flat_records(n_wg, items) <= w.rows, "%s", what);
                                    REQUIRE((size_t)groups * leap::counters_per_group(n_wg) <= w.counter_ints, "%s", what);
                                }
                    }
    REQUIRE(flat > 1000 && flat_partial > 1000 && split_views > 1000, "flat %lld, of a part of the handle %lld, split views %lld",
            flat, flat_partial, split_views);
    std::printf("calls %lld, flat %lld ok\n", calls, flat);
}
