// Row tiles of the attention kernels whose loops attn_loops.py writes (head dim 128, 16 bits, 16x16x32 MFMAs).
#pragma once
#include "attn_tile.h"

namespace dh {

// Tiles of 256-byte rows: the 16-byte chunk index of a row is XORed with swz16(row).  Row fragments (16 lanes = one chunk of 16
// consecutive rows) and transpose reads (32 lanes = 8 rows x 2 neighbouring chunks) are free of bank conflicts.
__device__ __forceinline__ int swz16(int row) { return 4 * (row & 3) + 2 * ((row >> 2) & 1) + ((row >> 3) & 1); }

// Raw buffer descriptor of rows, up to 4 GiB of wave-uniform address: the lanes of a copy that lie at or past `bytes` bring zeros.
__device__ __forceinline__ int4v rows_rsrc(const void *base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return int4v{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xffffu), (int)bytes, 0x00020000};
}
// Lane offsets of the 1 KB copies of 16 such rows, four rows each.
__device__ __forceinline__ void rows_lanes(uint32_t (&off)[4], int lane, uint32_t row_bytes) {
  const uint32_t row = (uint32_t)lane >> 4, chunk = ((uint32_t)lane & 15) ^ (4 * row);
#pragma unroll
  for (uint32_t x = 0; x < 4; ++x) off[x] = (4 * x + row) * row_bytes + ((chunk ^ (uint32_t)swz16(4 * x)) << 4);
}
// 64 lanes x 4 bytes, as copy_1k.
__device__ __forceinline__ void copy_256(uint32_t lane_off, const int4v &rsrc, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dword %0, %1, 0 offen lds" : : "v"(lane_off), "s"(rsrc), "s"(dst) : "memory", "m0");
}

// What a workgroup of a grid of (tiles of the longest sequence, or pairs of them, x heads, sequences) works on: the workgroups with work come
// first, those of the longest sequences ahead (batches of up to 64), and where the last of a head's pairs is only half of one, the same pair of several
// heads follow each other.  Workgroups go to the four shader engines of an XCD in turn, whatever they turn out to do: in the order of a grid laid
// out for the longest sequence every second one was often none or half as long, and half of the engines idled.  Forward, us, 32 query / 8 kv heads, causal, 24 sequences of 207 to 619 rows
// 227 -> 152, 8 x 527 to 1580 246 -> 184, 24 x 755 (three tiles: a pair and a half) 306 -> 256.
struct RowWork {
  int b, hkv, h, px;   // b < 0: nothing
};
template <int BM> __device__ __forceinline__ RowWork row_work(const int32_t *cu, int shift, int max_sq, int hq, int hk, int causal) {
  const int n = gridDim.y, lane = threadIdx.x & 63, ratio = hq / hk;
  auto length = [&](int i) { return (cu[i + 1] >> shift) - (cu[i] >> shift); };
  auto items = [&](int len) {
    const int t = (min(len, max_sq) + BM - 1) / BM;
    return causal ? (t + 1) / 2 : t;
  };
  int b = blockIdx.y, id = blockIdx.x, len, P;
  if (n == 1 || n > 64) {
    len = length(b);
    P = items(len);
    if (id >= P * hq) return {-1, 0, 0, 0};
  } else {
    // lane j: sequence j, its workgroups and where they end in the order of falling length (ties: lower index first)
    const int own = lane < n ? length(lane) : -1;
    len = __builtin_amdgcn_readfirstlane(own);
    P = items(len);
    if (__all(own == len || lane >= n)) {
      if (id >= P * hq) return {-1, 0, 0, 0};
    } else {
      const int count = lane < n ? items(own) * hq : 0;
      int end = 0;
#pragma unroll 4
      for (int j = 0; j < n; ++j) {
        const int o = __builtin_amdgcn_readlane(own, j), c = __builtin_amdgcn_readlane(count, j);
        end += o > own || (o == own && j <= lane) ? c : 0;
      }
      id += (int)(blockIdx.y * gridDim.x);
      const uint64_t mine = __ballot(id < end && id >= end - count);
      if (mine == 0) return {-1, 0, 0, 0};
      b = (int)__builtin_ctzll(mine);
      len = __builtin_amdgcn_readlane(own, b);
      P = items(len);
      id -= __builtin_amdgcn_readlane(end - count, b);
    }
  }
  const bool uneven = causal && (((min(len, max_sq) + BM - 1) / BM) & 1);
  if ((hk & 7) == 0) {
    const int x = id & 7, i = id >> 3;
    int at = i / P, px = i - at * P;                   // of the XCD's heads
    if (uneven) {
      const int heads = hq / 8, some = ratio >= 4 ? ratio : min(heads, 4), first = at / some * some, now = min(heads - first, some), in = i - first * P;
      px = in / now;
      at = first + in - px * now;
    }
    const int group = at / ratio;
    return {b, x + 8 * group, 8 * ratio * group + x * ratio + (at - group * ratio), px};
  }
  int hkv, item;
  xcd_group_item(id, hk, ratio * P, hkv, item);
  const int by = uneven ? ratio : P, q = item / by, m = item - q * by;
  return {b, hkv, hkv * ratio + (uneven ? m : q), uneven ? q : m};
}

}  // namespace dh
