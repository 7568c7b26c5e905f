// Grid sizes that the host can check without a device.
#pragma once
#include <cstdint>

namespace gsj {

// Blocks of 256 threads for n items (n > 0) of `lanes` threads each, numbered by flat_block(): up to 2^22 of them in a row,
// more in further rows. A launch holds fewer than 2^32 threads a dimension, as many as 2^28 items of 16 lanes in one row.
// (A loop over the items in one row of blocks cost the eroded self-join of 251k parcels 40 us of 2363, its two kernels'.)
struct ItemGrid { uint32_t x, y; };
inline ItemGrid item_grid(uint64_t n, uint32_t lanes) {
  const uint64_t row = 1u << 22, per = 256 / lanes, b = (n + per - 1) / per;
  return ItemGrid{(uint32_t)(b < row ? b : row), (uint32_t)((b + row - 1) / row)};
}

}  // namespace gsj
