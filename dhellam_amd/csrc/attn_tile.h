// Tile layout of the attention kernels that leave scheduling to the compiler (16 bits; all head dims, 128
// where its hand-ordered kernels are not the faster ones).
//
// A tile of 32 n rows of D elements lies in LDS without padding; the 16-byte chunk index of a row is XORed with swz(row).
// Both ways of reading are then free of bank conflicts:
//   * row fragments (ds_read_b128, 16 lanes = one chunk of 16 consecutive rows): where the row pitch 2 D puts 16 / n of the
//     rows on different multiples of 16 n bytes of the 256 that the banks span (n = 4 at D = 96, 8 at 64 and 192, 16 at
//     128 and 256), the XOR of the low log2(n) chunk bits tells the others apart: 16 different chunks;
//   * transpose reads (32 lanes = 4 consecutive rows x 4 neighbouring chunks): the pitch or bits 2 and 3 of the XOR put
//     the rows into the four 64-byte quarters of the banks, the chunks fill a quarter.
// Tiles are filled by global -> LDS copies of 1 KB per wavefront instruction with the swizzle on the global side; the
// pattern of rows and chunks repeats every 16 rows.
#pragma once
#include "mma.h"

namespace dh {

template <int D> struct AttnTile {
  static constexpr int CPR = D / 8, PITCH = 2 * D;                  // chunks and bytes of a row
  static constexpr int PAT = CPR / 4;                               // copies of 16 rows
  static constexpr int FIELD = D % 128 == 0 ? 15 : D % 64 == 0 ? 7 : 3;   // chunk bits that the swizzle touches
  static __device__ __forceinline__ int swz(int row) {
    return FIELD == 15 ? 4 * (row & 3) | ((row >> 2) & 3) : FIELD == 7 ? ((row >> 1) & 1) << 2 | ((row >> 2) & 3) : (row >> 2) & 3;
  }
};

// Largest token stride (elements of 16 bits) whose offsets across 15 rows fit the 32 bits of a lane's offset.
constexpr int64_t TILE_MAX_STRIDE = 1ll << 27;

// A wavefront's lane offsets for the copies of 16 rows.
template <int D> struct TileCopy { uint32_t off[AttnTile<D>::PAT]; };
template <int D> __device__ __forceinline__ void tile_copy_lane(int i, int lane, int &row, int &chunk) {
  using A = AttnTile<D>;
  const int l = 64 * i + lane;
  row = l / A::CPR;
  chunk = (l % A::CPR) ^ A::swz(row);
}
template <int D> __device__ __forceinline__ TileCopy<D> tile_copy(int lane, uint32_t row_bytes) {
  TileCopy<D> c;
#pragma unroll
  for (int i = 0; i < AttnTile<D>::PAT; ++i) {
    int row, chunk;
    tile_copy_lane<D>(i, lane, row, chunk);
    c.off[i] = (uint32_t)row * row_bytes + (uint32_t)chunk * 16;
  }
  return c;
}
// Rows row0 .. row0 + ROWS - 1 of `g` (ROWS and the tile row at `dst` multiples of 16) to LDS byte address `dst`; `rows`:
// rows of the sequence, later ones repeat the last; `whole`: the rows that the lane offsets reach (tile_whole_rows), others
// are addressed one by one.  The copies are not counted by the compiler (dma_wait_all).
__device__ __forceinline__ int tile_whole_rows(int rows, int64_t stride) { return stride <= TILE_MAX_STRIDE ? rows : 0; }
template <typename T, int D, int ROWS>
__device__ __forceinline__ void copy_tile(const T *g, int64_t stride, int row0, int rows, int whole, uint32_t dst, const TileCopy<D> &c, int lane) {
  constexpr int PAT = AttnTile<D>::PAT;
  if (row0 + ROWS <= whole) {
    const char *src = reinterpret_cast<const char *>(g + (int64_t)row0 * stride);
#pragma unroll
    for (int q = 0; q < ROWS / 16; ++q) {
#pragma unroll
      for (int i = 0; i < PAT; ++i) dma_block_fast(src, c.off[i], dst + 1024 * (q * PAT + i));
      src += 16 * stride * (int64_t)sizeof(T);
    }
  } else {
#pragma unroll 1
    for (int q = 0; q < ROWS / 16; ++q)
#pragma unroll
      for (int i = 0; i < PAT; ++i) {
        int row, chunk;
        tile_copy_lane<D>(i, lane, row, chunk);
        int r = row0 + 16 * q + row;
        r = r < rows ? r : rows - 1;
        const char *src = reinterpret_cast<const char *>(g + (int64_t)r * stride) + chunk * 16;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(dst + 1024 * (q * PAT + i)) : "memory", "m0");
      }
  }
}

// Loaded fragments that a loop only reads: the wait for them goes here.  Without this the compiler, which does not count the
// copies above, waits for them by "nothing outstanding" at their first use in every iteration, and so for the copies that
// were to run beneath it: a memory latency an iteration (forward of 16 heads x 2 x 512 at head dim 64 9.4 -> 8.0 us, backward 32
// query / 8 kv heads x 4096 328 -> 292).  More than two stages brought nothing beyond that (4: 298, 3: 297 us).
template <int N, typename F> __device__ __forceinline__ void loaded_here(F (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}

template <typename T> using lds_frag_t = __attribute__((address_space(3))) const typename Mma<T>::Frag *;
typedef short4v __attribute__((address_space(3))) *lds_tr_t;

// Row fragments: lane offset of row c (rows c + 32 n: + 32 n PITCH) and its chunk of k step 0; k step ks by row_frag().
struct RowLane { uint32_t base, x; };
template <int D> __device__ __forceinline__ RowLane row_lane(int lane) {
  const int c = lane & 31, hh = lane >> 5;
  return RowLane{(uint32_t)(c * AttnTile<D>::PITCH), (uint32_t)((hh ^ AttnTile<D>::swz(c)) << 4)};
}
template <typename T, int D> __device__ __forceinline__ typename Mma<T>::Frag row_frag(uint32_t tile, const RowLane &l, int ks) {
  constexpr int F = AttnTile<D>::FIELD;
  return *(lds_frag_t<T>)(tile + l.base + (l.x ^ (uint32_t)((2 * ks & F) << 4)) + (uint32_t)((2 * ks & ~F) << 4));
}
// Transposed fragments of 16 rows (k) x 32 columns: rows 4 hh + r / 4 and 8 further down, columns 16 ((lane / 16) % 2) +
// 4 (r % 4) of a 32-column block (r = lane % 16).
struct TrLane { uint32_t base, xa, xb; };
template <int D> __device__ __forceinline__ TrLane tr_lane(int lane) {
  using A = AttnTile<D>;
  const int r = lane & 15, row = 4 * (lane >> 5) + (r >> 2), chunk = 2 * ((lane >> 4) & 1) + ((r & 3) >> 1);
  return TrLane{(uint32_t)(row * A::PITCH + 8 * (r & 1)), (uint32_t)((chunk ^ A::swz(row)) << 4), (uint32_t)((chunk ^ A::swz(row + 8)) << 4)};
}
template <typename T, int D> __device__ __forceinline__ typename Mma<T>::Frag tr_frag(uint32_t tile, const TrLane &l, int t, int s) {
  using A = AttnTile<D>;
  const uint32_t at = tile + l.base + (uint32_t)(((4 * t & ~A::FIELD) << 4) + s * 16 * A::PITCH), f = (uint32_t)((4 * t & A::FIELD) << 4);
  const short4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + (l.xa ^ f)));
  const short4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + 8 * A::PITCH + (l.xb ^ f)));
  return frag_join<T>(x, y);
}

// Four consecutive values of a row of `T` in memory.
template <typename T> struct alignas(8) Quad { T v[4]; };

}  // namespace dh
