// Host-side check of the rules that size and route a launch, on the library's
// own source (no device): over every supported head shape, handles of 1-128
// sequences, fewer sequences than the handle holds, and row counts given or
// estimated, a flat launch's kernel exists and its records and counters fit
// in the handle's workspace; and batches on both sides of the rule's lines take
// the route that measured faster.  With "route" as its argument, it answers
// calls read from its input instead: q heads, KV heads, head_dim, seq_len,
// max_batch, sequences, the longest and all rows (0: not given) -> workgroups
// per XCD of the flat launch, 0 for a uniform one.  Built and run by
// tests/test_launch_rules.py.
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

namespace {

leap_hip_attention handle(int n_heads, int n_kv_heads, int head_dim, int seq_len, int max_batch, int n_cu)
{
    leap_hip_attention_config c{};
    c.n_layers = c.layer_end = 1;
    c.n_heads = n_heads;
    c.n_kv_heads = n_kv_heads;
    c.head_dim = head_dim;
    c.seq_len = seq_len;
    c.max_batch = max_batch;
    const Workspace w = workspace_for(c, n_cu);
    leap_hip_attention h;
    h.cfg = c;
    h.group = n_heads / n_kv_heads;
    h.n_cu = n_cu;
    h.max_chunks = w.max_chunks;
    h.max_flat = w.max_flat;
    return h;
}

int flat_workgroups(const leap_hip_attention &h, int n_seq, long long rows, int max_T)
{
    return flat_launch(launch_view(shape_of(&h), n_seq, rows), n_seq, rows, max_T);
}

// Batches of a full handle: q heads, KV heads, head_dim, sequences, the
// longest and all rows (0: not given), and whether flat measured faster.
const struct {
    int n_heads, n_kv_heads, head_dim, n_seq, max_T;
    long long rows;
    bool flat;
} kRoutes[] = {
    // equal lengths
    {32, 8, 128, 12, 2000, 12 * 2000, true},
    {32, 8, 128, 3, 4000, 3 * 4000, true},
    {32, 8, 128, 32, 1000, 32 * 1000, false},
    {64, 8, 128, 12, 2000, 12 * 2000, true},
    {64, 8, 128, 28, 500, 28 * 500, false},
    {128, 8, 128, 6, 2000, 6 * 2000, true},
    {128, 8, 128, 24, 500, 24 * 500, false},
    {32, 32, 128, 3, 2000, 3 * 2000, true},
    {16, 16, 64, 20, 200, 20 * 200, false},
    {32, 4, 64, 32, 1000, 32 * 1000, true},
    {32, 4, 64, 8, 1000, 8 * 1000, false},
    {32, 4, 64, 28, 1000, 28 * 1000, true},
    {32, 4, 64, 28, 200, 28 * 200, false},
    // one or two rows short of the longest
    {32, 8, 128, 12, 2000, 12 * 2000 - 12, true},
    {32, 8, 128, 32, 200, 32 * 200 - 31, false},
    {32, 8, 128, 32, 1000, 32 * 1000 - 31, false},
    {32, 8, 128, 8, 4000, 8 * 4000 - 7, false},
    {32, 8, 128, 2, 4000, 2 * 4000 - 1, false},
    {24, 8, 128, 32, 500, 32 * 500 - 31, false},
    {64, 8, 128, 32, 1000, 32 * 1000 - 31, false},
    {64, 8, 128, 24, 2000, 24 * 2000 - 24, true},
    {128, 8, 128, 16, 200, 16 * 200 - 15, false},
    {32, 16, 128, 16, 500, 16 * 500 - 15, false},
    {32, 4, 64, 32, 1000, 32 * 1000 - 31, true},
    // ragged
    {32, 8, 128, 16, 2011, 16 * 1100, true},
    {32, 8, 128, 64, 8192, 64 * 4300, true},
    {64, 8, 128, 16, 2000, 16 * 1100, true},
    {32, 8, 128, 24, 300, 24 * 160, false},
    {32, 8, 128, 16, 2011, 0, true},
    {32, 8, 64, 4, 2000, 3869, true},
    {32, 8, 64, 8, 1000, 0, true},
    {32, 8, 64, 48, 130, 48 * 80, false},
};

}  // namespace

int main(int argc, char **)
{
    if (argc > 1) {
        int nh, nkv, hd, seq_len, max_batch, n_seq, max_T;
        long long rows;
        while (std::scanf("%d %d %d %d %d %d %d %lld", &nh, &nkv, &hd, &seq_len, &max_batch, &n_seq, &max_T, &rows) == 8)
            std::printf("%d\n", flat_workgroups(handle(nh, nkv, hd, seq_len, max_batch, 256), n_seq,
                                                rows > 0 ? rows : rows_estimate(n_seq, max_T), max_T));
        return 0;
    }
    for (const auto &r : kRoutes) {
        const long long rows = r.rows > 0 ? r.rows : rows_estimate(r.n_seq, r.max_T);
        const int n_wg = flat_workgroups(handle(r.n_heads, r.n_kv_heads, r.head_dim, r.max_T, r.n_seq, 256), r.n_seq, rows, r.max_T);
        REQUIRE((n_wg > 0) == r.flat, "heads %d/%d/%d, %d sequences, longest %d, rows %lld: %d workgroups per XCD", r.n_heads,
                r.n_kv_heads, r.head_dim, r.n_seq, r.max_T, r.rows, n_wg);
    }
    long long calls = 0, flat = 0, flat_partial = 0, split_views = 0;
    for (int n_cu : {256, 128, 64, 32})
        for (int hd : {64, 128})
            for (int g : {1, 2, 3, 4, 8, 16})
                for (int nkv : {1, 2, 3, 4, 5, 8, 10, 16, 32, 40})
                    for (int max_batch : {1, 2, 3, 4, 5, 8, 16, 33, 64, 128}) {
                        const leap_hip_attention h = handle(g * nkv, nkv, hd, 32768, max_batch, n_cu);
                        const Workspace w = workspace_for(h.cfg, n_cu);
                        std::set<int> ns;
                        for (int n : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64, 100, 128}) ns.insert(std::min(n, max_batch));
                        for (int n_seq : ns)
                            for (int max_T : {1, 31, 64, 100, 500, 1000, 1024, 2011, 3000, 4095, 4096, 5000, 6143, 8192,
                                              12288, 16384, 24576, 32768})
                                // estimated (total_rows 0), equal lengths, ragged ones, one long among short
                                for (long long rows : {rows_estimate(n_seq, max_T), (long long)n_seq * max_T,
                                                       (long long)n_seq * max_T * 5 / 6, (long long)max_T + n_seq - 1}) {
                                    calls++;
                                    const LaunchShape s = launch_view(shape_of(&h), n_seq, rows);
                                    if (s.kv_split != shape_of(&h).kv_split) split_views++;
                                    const int n_wg = flat_workgroups(h, n_seq, rows, max_T);
                                    if (!n_wg) continue;
                                    flat++;
                                    flat_partial += n_seq < max_batch;
                                    char what[160];
                                    std::snprintf(what, sizeof what, "%d CUs, heads %d/%d/%d, %d of %d sequences, longest %d, rows %lld",
                                                  n_cu, h.cfg.n_heads, nkv, hd, n_seq, max_batch, max_T, rows);
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
