// pack.hpp — the weight packing launch of pack.hip, called by the C ABI.
#pragma once

#include <stdint.h>

namespace bsgk {

// Checked arguments of bsg_pack_weight; 0, a hipError_t, or -1 when the grid would be too large.
int launch_pack(const void* w, int64_t N, int64_t K, int64_t stride_n, int64_t stride_k, void* wp, void* stream);

}  // namespace bsgk
