// fp32 projection GEMV instances (see kernels.hpp).
#include "kernels.hpp"

namespace leap_kernels {

// An fp32 projection kernel by width 1024 * NC and rows per workgroup RB.  A
// launch takes the RB that leaves the busiest CU the fewest rows, the larger
// one on a tie: workgroups that are not a whole number per CU leave CUs idle
// for the last of them.  Up to 32 / NC rows (128 KiB of weights in flight per
// workgroup; at Llama-3-8B 64 KiB and 256 KiB measured slower), 12 at 3072,
// where the wo product's 3072 rows then make one workgroup per CU.  us per
// launch, back to back over 1.6 GiB of weights, at 32 / NC rows -> now:
// TinyLlama q/k/v (2560 rows of 2048; 160 workgroups of 16 -> 256 of 10) 5.56
// -> 4.81, wo (2048; 128 of 16 -> 256 of 8) 5.23 -> 4.50; Llama-3.2-3B wo
// (3072; 308 of 10 -> 256 of 12) 8.78 -> 7.40; Llama-2-13B wo (5120; 854 of 6
// -> 1024 of 5) 17.78 -> 17.13; Llama-3-70B q/k/v (10240; 2560 of 4 -> 2048
// of 5) 49.55 -> 49.12.
struct ProjEntry {
    int dim, rb;
    QkvFn qkv;
    ProjFn proj;
    GemvFloorFn floor;
};
#define LEAP_PROJ(NC, RB) \
    {1024 * NC, RB, leap::qkv_kernel<RB, NC>, leap::proj_residual_kernel<RB, NC>, leap::gemv_floor_kernel<RB, NC>},
const ProjEntry kProjKernels[] = {
    LEAP_PROJ(2, 16) LEAP_PROJ(2, 12) LEAP_PROJ(2, 10) LEAP_PROJ(2, 8)
    LEAP_PROJ(3, 12) LEAP_PROJ(3, 10)
    LEAP_PROJ(4, 8) LEAP_PROJ(4, 6)
    LEAP_PROJ(5, 6) LEAP_PROJ(5, 5)
    LEAP_PROJ(8, 5) LEAP_PROJ(8, 4)
};
#undef LEAP_PROJ

bool pick_proj(int dim, int rows, int n_cu, ProjLaunch *out)
{
    const ProjEntry *best = nullptr;
    long long best_rows = 0;  // rows of the busiest CU
    for (const ProjEntry &k : kProjKernels) {
        if (k.dim != dim) continue;
        const long long wgs = (rows + k.rb - 1) / k.rb, most = (wgs + n_cu - 1) / n_cu * k.rb;
        if (!best || most < best_rows || (most == best_rows && k.rb > best->rb)) {
            best = &k;
            best_rows = most;
        }
    }
    if (!best) return false;
    *out = ProjLaunch{best->qkv, best->proj, best->floor, (rows + best->rb - 1) / best->rb};
    return true;
}

}  // namespace leap_kernels
