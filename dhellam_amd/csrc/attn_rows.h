// Row tiles of the attention kernels whose loops attn_loops.py writes (head dim 128, 16 bits, 16x16x32 MFMAs).
#pragma once
#include "attn_tile.h"

namespace dh {

typedef int int4s __attribute__((ext_vector_type(4)));

// Tiles of 256-byte rows: the 16-byte chunk index of a row is XORed with swz16(row).  Row fragments (16 lanes = one chunk of 16
// consecutive rows) and transpose reads (32 lanes = 8 rows x 2 neighbouring chunks) are free of bank conflicts.
__device__ __forceinline__ int swz16(int row) { return 4 * (row & 3) + 2 * ((row >> 2) & 1) + ((row >> 3) & 1); }

// Raw buffer descriptor of rows that may reach past the end: the lanes of a copy that lie at or past `bytes` bring zeros.
__device__ __forceinline__ int4s rows_rsrc(const void *base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return int4s{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xffffu), (int)bytes, 0x00020000};
}
// Lane offsets of the 1 KB copies of 16 such rows, four rows each.
__device__ __forceinline__ void rows_lanes(uint32_t (&off)[4], int lane, uint32_t row_bytes) {
  const uint32_t row = (uint32_t)lane >> 4, chunk = ((uint32_t)lane & 15) ^ (4 * row);
#pragma unroll
  for (uint32_t x = 0; x < 4; ++x) off[x] = (4 * x + row) * row_bytes + ((chunk ^ (uint32_t)swz16(4 * x)) << 4);
}
// 64 lanes x 16 (or 4) bytes from descriptor base + lane offset + `off` to LDS byte address `dst`, which the compiler does not
// count among what is in flight.
__device__ __forceinline__ void copy_1k(uint32_t lane_off, const int4s &rsrc, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(lane_off), "s"(rsrc), "s"(off), "s"(dst)
               : "memory", "m0");
}
__device__ __forceinline__ void copy_256(uint32_t lane_off, const int4s &rsrc, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" : : "v"(lane_off), "s"(rsrc), "s"(dst) : "memory", "m0");
}

}  // namespace dh
