// dequant_plan.h -- how the dequantiser's launches divide its super-blocks.
// Plain host arithmetic, in a header of its own so that the host tests compile
// the same rule.
#pragma once

#include <stdint.h>

namespace iq4xs {

constexpr int64_t DEQUANT_THREADS = 32;  // per super-block
constexpr int64_t DEQUANT_WG = 256;      // threads per workgroup

// Super-blocks of the next launch when `left` remain.  A launch of HIP holds
// fewer than 2^32 threads, so one takes at most 2^27 - 8 super-blocks (128 GiB
// of output): a larger call is several launches.
constexpr int64_t dequant_chunk(int64_t left) {
    constexpr int64_t kMax = (((int64_t)1 << 32) - DEQUANT_WG) / DEQUANT_THREADS;
    return left < kMax ? left : kMax;
}

}  // namespace iq4xs
