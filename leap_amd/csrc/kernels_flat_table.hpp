// The flat decode kernel's instances for one head_dim, included by the
// kernels_decode_*f.hip translation units only.
#pragma once

#include "kernels.hpp"

namespace leap_kernels {

template <int HD>
KernelFn pick_flat(int g, int kvs)
{
    if (kvs) return kvs == 1 && g == 8 ? leap::decode_attention_flat_kernel<HD, 8, kWaves, 1> : nullptr;
#define LEAP_CASE(G) \
    if (g == G) return leap::decode_attention_flat_kernel<HD, G, kWaves, 0>;
    LEAP_CASE(1) LEAP_CASE(2) LEAP_CASE(3) LEAP_CASE(4) LEAP_CASE(8)
#undef LEAP_CASE
    return nullptr;
}

}  // namespace leap_kernels
