// Grid sizes that the host can check without a device.
#pragma once
#include <cstdint>

namespace gsj {

// Blocks of 256 threads for n items of `lanes` threads each (n > 0), taken by stride: one round up to 2^22 blocks, several
// beyond. A launch holds fewer than 2^32 threads a dimension, and 2^28 items of 16 lanes would be as many.
constexpr uint32_t STRIDE_BLOCKS = 1u << 22;
inline uint32_t stride_blocks(uint64_t n, uint32_t lanes) {
  const uint64_t per = 256 / lanes, b = (n + per - 1) / per;
  return b < STRIDE_BLOCKS ? (uint32_t)b : STRIDE_BLOCKS;
}

}  // namespace gsj
