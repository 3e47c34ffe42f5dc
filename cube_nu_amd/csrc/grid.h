// grid.h -- launches whose threads along x would pass 2^32.
#pragma once
#include <algorithm>
#include <cstdint>

namespace cube {

// A launch dimension holds fewer than 2^32 threads, so blocks beyond 2^21 (of at
// most 1024 threads) go on along y; block (x, y) is y * gridDim.x + x, and a kernel
// drops those past its last.
struct Blocks {
  uint32_t x, y;
};
constexpr int64_t kBlocksX = (int64_t)1 << 21;
constexpr Blocks blocks_xy(int64_t blocks) {
  return blocks <= kBlocksX ? Blocks{(uint32_t)blocks, 1}
                            : Blocks{(uint32_t)kBlocksX, (uint32_t)((blocks + kBlocksX - 1) / kBlocksX)};
}

// The other way: n items in pieces of at most `most`, fn(first, items) a launch each.
template <class Fn>
inline void in_pieces(int64_t n, int64_t most, Fn&& fn) {
  for (int64_t at = 0; at < n; at += most) fn(at, std::min(n - at, most));
}

}  // namespace cube
