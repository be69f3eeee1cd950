// The order in which workgroups take the tiles of a matrix product.
#pragma once
#include "common.h"

namespace dh {

// Workgroup ids go round the 8 XCDs; this gives XCD x (the ids x, x + 8, ...) the x-th of 8 contiguous chunks of
// 0..n-1, so that neighbouring tiles share an L2 (a bijection for any n: the first n % 8 chunks are one longer).
__device__ __forceinline__ int gg_xcd_chunk(int id, int n) {
  const int q8 = n / 8, r8 = n % 8, x = id % 8;
  return x * q8 + (x < r8 ? x : r8) + id / 8;
}

// Tile t of the list -> (m tile, n tile): bands of 8 m tiles, m fastest inside a band, so that the 32 tiles an XCD has in
// flight are 8 x 4 and share 12 operand panels through its L2 instead of 18 + 2 (1-2 % on the FFN products).
__device__ __forceinline__ void gg_tile_of(int t, int tiles_m, int tiles_n, int &tm, int &tn) {
  constexpr int GM = 8;
  const int band = t / (GM * tiles_n), first = band * GM, gm = min(GM, tiles_m - first), in_band = t - band * GM * tiles_n;
  tm = first + in_band % gm;
  tn = in_band / gm;
}

}  // namespace dh
