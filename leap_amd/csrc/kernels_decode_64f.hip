// Flat decode-attention instances at head_dim 64 (see kernels.hpp).
#include "kernels_flat_table.hpp"

namespace leap_kernels {
template KernelFn pick_flat<64>(int, int);
}  // namespace leap_kernels
