// int8 W8A8 projection GEMV instances (see kernels.hpp).
#include "kernels.hpp"

namespace leap_kernels {

// The int8 projection kernels by width n = NL * 1024, lanes per group L =
// gs/16, rows per team J, waves NWV, waves per team WPR and input kind.  J and
// NWV are compiled in (every load of a thread is then unconditional); a launch
// takes the smallest instance that covers its rows with the fewest workgroups
// per CU.
struct Q8Entry {
    int nl, l, rows, threads, kind;
    Q8Fn fn;
    Q8Fn floor;  // the same grid streaming the weights alone (measurement)
};

// The sizes of a width: the rows per CU of the models that have it, and what
// lies between.  Rows per CU (q/k/v, wo): TinyLlama 10, 8; Llama-3.2-3B 20,
// 12; Llama-3-8B 24, 16; Llama-2-7B 48, 16; Llama-2-13B 60, 20; Llama-3-70B
// 40, 32.  Measured around them, us per launch: 24 rows as 8 waves x 3 6.35,
// 12 x 2 6.68, 6 x 4 6.78, 16 (teams of 2) x 3 7.01; 10 rows as 5 x 2 2.94,
// 10 x 1 3.19; 60 rows as 12 x 5 16.5, 10 x 6 16.8, 6 x 10 21.8; 20 rows at
// 5120 as 10 x 2 7.04, 5 x 4 7.49; 40 rows at 8192 as 16 waves in teams of 2
// x 5 17.2, 8 x 5 17.8, 10 x 4 25.7.  Rows per CU between two sizes leave slots
// idle (5120 with 10 KV heads: 30 of 60), which still beats a team per row:
// its sub-block 26.7 -> 24.3.
#define LEAP_Q8_K(NL, L, J, NWV, WPR, K)                                                                \
    {NL, L, J * NWV / WPR, NWV * 64, K, leap::q8_gemv_kernel<NL, L, J, NWV, WPR, K, K != leap::kQ8InRms>, \
     leap::q8_floor_kernel<NL, L, J, NWV, WPR>},
#define LEAP_Q8(NL, L, J, NWV, WPR) LEAP_Q8_K(NL, L, J, NWV, WPR, leap::kQ8InRms) LEAP_Q8_K(NL, L, J, NWV, WPR, leap::kQ8InF32)
#define LEAP_Q8_2048(L) LEAP_Q8(2, L, 1, 8, 1) LEAP_Q8(2, L, 2, 5, 1) LEAP_Q8(2, L, 2, 8, 1) LEAP_Q8(2, L, 3, 8, 1)
#define LEAP_Q8_3072(L) LEAP_Q8(3, L, 2, 6, 1) LEAP_Q8(3, L, 4, 5, 1) LEAP_Q8(3, L, 3, 12, 1)
#define LEAP_Q8_4096(L) LEAP_Q8(4, L, 2, 8, 1) LEAP_Q8(4, L, 3, 8, 1) LEAP_Q8(4, L, 3, 16, 1)
#define LEAP_Q8_5120(L) LEAP_Q8(5, L, 2, 10, 1) LEAP_Q8(5, L, 5, 12, 1)
#define LEAP_Q8_8192(L) LEAP_Q8(8, L, 4, 16, 2) LEAP_Q8(8, L, 5, 16, 2)
const Q8Entry kQ8Kernels[] = {
    LEAP_Q8_2048(2) LEAP_Q8_2048(4) LEAP_Q8_2048(8)
    LEAP_Q8_3072(2) LEAP_Q8_3072(4) LEAP_Q8_3072(8)
    LEAP_Q8_4096(2) LEAP_Q8_4096(4) LEAP_Q8_4096(8) LEAP_Q8_4096(16)
    LEAP_Q8_5120(4) LEAP_Q8_5120(8)
    LEAP_Q8_8192(4) LEAP_Q8_8192(8) LEAP_Q8_8192(16)
};
#undef LEAP_Q8_8192
#undef LEAP_Q8_5120
#undef LEAP_Q8_4096
#undef LEAP_Q8_3072
#undef LEAP_Q8_2048
#undef LEAP_Q8
#undef LEAP_Q8_K

// True if (dim, gs) has int8 kernels.
bool q8_supported(int dim, int gs)
{
    for (const Q8Entry &k : kQ8Kernels)
        if (k.nl * 1024 == dim && k.l * 16 == gs) return true;
    return false;
}

bool pick_q8(int dim, int gs, int kind, int rows, int n_cu, Q8Launch *out)
{
    const int need = (rows + n_cu - 1) / n_cu;  // rows per CU
    const Q8Entry *best = nullptr;
    int best_per_cu = 0;  // workgroups per CU
    for (const Q8Entry &k : kQ8Kernels) {
        if (k.nl * 1024 != dim || k.l * 16 != gs || k.kind != kind) continue;
        const int per_cu = (need + k.rows - 1) / k.rows;
        if (!best || per_cu < best_per_cu || (per_cu == best_per_cu && k.rows < best->rows)) {
            best = &k;
            best_per_cu = per_cu;
        }
    }
    if (!best) return false;
    out->fn = best->fn;
    out->floor = best->floor;
    out->per_wg = (need + best_per_cu - 1) / best_per_cu;
    out->grid = (rows + out->per_wg - 1) / out->per_wg;
    out->threads = best->threads;
    return true;
}

}  // namespace leap_kernels
