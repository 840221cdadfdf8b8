// sa_tile_place.hpp -- which tile of which system a block of a tile sweep works on, and how
// many systems a launch can have.
#pragma once

#include <algorithm>
#include <cstdint>

namespace sa {

struct tile_place {
  uint32_t sys, bx, by;
};

// ceil(2^32 / per): per = tiles of a system (not used with one)
constexpr uint32_t tile_recip(uint32_t per) { return (uint32_t)((((uint64_t)1 << 32) + per - 1) / per); }

// quotient of small non-negative integers (n * (d - 1) < 2^20), from ceil(2^20 / d)
constexpr int small_recip(int d) { return ((1 << 20) + d - 1) / d; }
constexpr int small_div(int n, int d_recip20) { return (int)(((uint32_t)n * (uint32_t)d_recip20) >> 20); }

// Tile b of all systems' tiles, system by system, rows of ntx tiles.
constexpr tile_place place_tile(uint32_t b, uint32_t per, uint32_t recip_per, uint32_t ntx, int recip_ntx) {
  const uint32_t sys = per == 1 ? b : (uint32_t)(((uint64_t)b * recip_per) >> 32), r = b - sys * per;
  const uint32_t by = (uint32_t)small_div((int)r, recip_ntx);
  return tile_place{sys, r - by * ntx, by};
}

// Systems one launch can take, of `per` blocks of `threads` each (rounded up to 8 blocks): a
// launch has fewer than 2^32 threads, and the reciprocal above is exact for b * x < 2^32 where x
// = per * recip_per - 2^32.  A larger ladder takes several launches (odd 3D L=247, 3844 tiles:
// 360 systems each; correcting the quotient in the kernel instead cost 0.5% at L=64).
constexpr int64_t systems_per_launch(uint32_t per, int threads) {
  const int64_t by_grid = (((int64_t)1 << 32) - 1) / threads - 8;
  const int64_t x = per == 1 ? 0 : (int64_t)((uint64_t)per * tile_recip(per) - ((uint64_t)1 << 32));
  const int64_t by_recip = x == 0 ? by_grid : (((int64_t)1 << 32) - 1) / x;
  return std::min(by_grid, by_recip) / per;
}

}  // namespace sa
