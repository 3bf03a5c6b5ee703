// Flat decode-attention instances at head_dim 128 (see kernels.hpp).
#include "kernels_flat_table.hpp"

namespace leap_kernels {
template KernelFn pick_flat<128>(int, int);
}  // namespace leap_kernels
