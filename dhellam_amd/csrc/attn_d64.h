// Head-dim-64 attention kernels (16 bits): shared tile layout.
//
// A tile of 64-element rows lies in LDS as 256-byte lines of two rows each; the 16-byte chunk index of a line (bit 3: odd
// row) is XORed with line_swz(line).  Both ways of reading are then free of bank conflicts:
//   * row fragments (ds_read_b128; 16 lanes = 16 consecutive rows = 8 lines x 2 halves): line_swz is a bijection of
//     line % 8 in the low three chunk bits, bit 3 is the row's parity: 16 different chunks;
//   * transpose reads (32 lanes = 4 consecutive rows x 4 chunks): the two lines differ in bit 2 of line_swz, the two rows
//     of a line in bit 3, the four chunks in bits 0-1.
// Tiles are filled by global -> LDS copies of 1 KB (8 rows) per wavefront instruction with the swizzle on the global side.
#pragma once
#include "mma.h"

namespace dh {

__device__ __forceinline__ int line_swz(int line) { return ((line & 1) << 2) | ((line >> 1) & 3); }

// Copies of one wavefront: CB consecutive 1 KB blocks (8 rows each) of one tile.
struct Copy64 {
  uint32_t off[2];       // lane byte offset from the first row of an even / odd block
  int row, ch[2];        // row inside the block, 16-byte chunk of the row in an even / odd block
};
__device__ __forceinline__ Copy64 copy64_lane(int lane, uint32_t row_bytes) {
  Copy64 c;
  const int x = (lane & 15) ^ (((lane >> 4) & 1) << 2) ^ (lane >> 5);
  c.row = 2 * (lane >> 4) + (x >> 3);
  c.ch[0] = x & 7;
  c.ch[1] = (x & 7) ^ 2;
  c.off[0] = (uint32_t)c.row * row_bytes + (uint32_t)c.ch[0] * 16;
  c.off[1] = (uint32_t)c.row * row_bytes + (uint32_t)c.ch[1] * 16;
  return c;
}
// Rows row0 .. row0 + 8 CB - 1 of `g` (row0 a multiple of 16) to LDS byte address `dst`; `rows`: rows of the sequence, later
// ones repeat the last.  The copies are not counted by the compiler (dma_wait_all).
template <typename T, int CB>
__device__ __forceinline__ void copy64(const T *g, int64_t stride, int row0, int rows, uint32_t dst, const Copy64 &c) {
  if (row0 + 8 * CB <= rows) {
    const char *src = reinterpret_cast<const char *>(g + (int64_t)row0 * stride);
    const uint32_t step = (uint32_t)(8 * stride * (int64_t)sizeof(T));
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      dma_block_fast(src, c.off[i & 1], dst + 1024 * i);
      src += step;
    }
  } else {
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      int r = row0 + 8 * i + c.row;
      r = r < rows ? r : rows - 1;
      const char *src = reinterpret_cast<const char *>(g + (int64_t)r * stride) + c.ch[i & 1] * 16;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(dst + 1024 * i) : "memory", "m0");
    }
  }
}

template <typename T> using lds_frag_t = __attribute__((address_space(3))) const typename Mma<T>::Frag *;
typedef short4v __attribute__((address_space(3))) *lds_tr_t;

// Lane byte offset of the row fragment of chunk hh of row c (rows c + 32 n: + 4096 n; k step ks: ^ (ks << 5)).
__device__ __forceinline__ uint32_t row64_lane(int lane) {
  const int c = lane & 31, hh = lane >> 5;
  return (uint32_t)((c >> 1) * 256 + (((((c & 1) << 3) | hh) ^ line_swz(c >> 1)) << 4));
}
// Lane byte offset of the transpose read of rows 4 hh + r / 4, columns 16 ((lane / 16) % 2) + 4 (r % 4) (r = lane % 16):
// 32-column block t: ^ (t << 6); rows + 16 s: + 2048 s; the rows 8 further down: tr64_next().
__device__ __forceinline__ uint32_t tr64_lane(int lane) {
  const int r = lane & 15, hh = lane >> 5;
  const int chunk = 2 * ((lane >> 4) & 1) + ((r & 3) >> 1);
  return (uint32_t)((2 * hh + (r >> 3)) * 256 + ((((((r >> 2) & 1) << 3) | chunk) ^ (((r >> 3) << 2) | hh)) << 4) + 8 * (r & 1));
}
__device__ __forceinline__ uint32_t tr64_next(uint32_t a) { return (a ^ 32u) + 1024u; }

template <typename T> __device__ __forceinline__ typename Mma<T>::Frag row64(uint32_t at) { return *(lds_frag_t<T>)(at); }
template <typename T> __device__ __forceinline__ typename Mma<T>::Frag tr64(uint32_t a, uint32_t b) {
  const short4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(a));
  const short4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(b));
  return frag_join<T>(x, y);
}

// Four consecutive values of a row of `T` in memory.
template <typename T> struct alignas(8) Quad { T v[4]; };

}  // namespace dh
