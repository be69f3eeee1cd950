// Dense products of fp32 matrices where the library's tiles leave the fp32 matrix pipe idle.
#include "gemm_f32.h"
#include "mma.h"
#include "tile_order.h"

namespace dh {

// One operand of a tile: 64 rows of X (or columns of Y) by slices of 32 along k, 8 KB each in LDS.
//   k contiguous: [64][32], 16-byte chunk XOR (row / 2) % 8: 16 rows' reads of one chunk hit 16 different chunks of 256 bytes; a lane
//     reads four consecutive k of its row at once.
//   k strided: [32][64], 16-byte chunk XOR 4 (k / 4 % 4): the four k rows that 64 lanes read lie in four different quarters of them.
// MFMA i of a step of 16 k multiplies k = 4 g + i on the lanes of group g, in both layouts.
template <bool STRIDED> struct F32Side {
  static constexpr uint32_t CROWS = STRIDED ? 4 : 8;              // rows of LDS a 1 KB copy
  const char *base;                                               // of the tile's slice 0
  int64_t step, len;                                              // from slice to slice; bytes behind base that may be read of slice 0
  uint32_t lane_off, off[2];                                      // a wavefront's two copies of a slice

  __device__ __forceinline__ F32Side(const float *ptr, int64_t first, int64_t extent, int64_t k, int wq, int lane) {
    const uint32_t ldb = 4u * (uint32_t)(STRIDED ? extent : k);
    if constexpr (STRIDED) {
      base = reinterpret_cast<const char *>(ptr + first);
      step = 32ll * ldb;
      len = (k - 1) * ldb + (extent - first) * 4;
      lane_off = (uint32_t)(lane >> 4) * ldb + (uint32_t)((lane & 15) ^ (4 * wq)) * 16u;
    } else {
      base = reinterpret_cast<const char *>(ptr + first * k);
      step = 128;
      len = ((extent - first < 64 ? extent - first : 64) - 1) * ldb + 128;
      lane_off = (uint32_t)(lane >> 3) * ldb + (uint32_t)((lane & 7) ^ (((lane >> 4) & 3) | (4 * (wq & 1)))) * 16u;
    }
    off[0] = (uint32_t)wq * CROWS * ldb;
    off[1] = (uint32_t)(wq + 4) * CROWS * ldb;
  }
  __device__ __forceinline__ int4v slice(int s, int nsl) const { return raw_rsrc(base + s * step, s >= nsl ? 0 : STRIDED ? len - s * step : len); }
};

template <bool STRIDED> struct F32Reads {
  typedef __attribute__((address_space(3))) const float *lds_f;
  typedef __attribute__((address_space(3))) const floatx4 *lds_f4;
  uint32_t at[2];                                                 // strided: of a block; else of a step
  __device__ __forceinline__ F32Reads(int first, int lane) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (STRIDED) at[i] = (uint32_t)(4 * g * 256 + (((((first + 16 * i + r) >> 2) ^ (4 * g)) << 4) | ((r & 3) << 2)));
      else at[i] = (uint32_t)((first + r) * 128 + (((4 * i + g) ^ ((r >> 1) & 7)) << 4));
    }
  }
  // block `b` of 16, step j of the slice
  __device__ __forceinline__ floatx4 get(uint32_t side, int b, int j) const {
    if constexpr (STRIDED) {
      floatx4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *(lds_f)(side + at[b] + (uint32_t)((16 * j + i) * 256));
      return v;
    } else {
      return *(lds_f4)(side + at[j] + (uint32_t)(b * 16 * 128));
    }
  }
};

// A workgroup of four wavefronts makes a tile of 64 x 64 (2 x 2 of 32 x 32), in slices of 32 along k that come to LDS by copies in three
// stages: 48 KB, so that three workgroups share a compute unit.  Fragments are read one step of 16 k ahead of their MFMAs, so that the one
// barrier of a slice stands in front of its last step: behind it everyone has the next slice, and has read all of this one, whose stage the
// copies of the third next take.  A 16x16x4 MFMA
// holds the matrix pipe for 32 cycles: reads and copies go between them, and the loop's code has nothing else.
// What bounds it is the path from L2: 16 KB a slice, 8 TB/s at 85 % of the pipe's rate (256 tiles, one a compute unit, 7 TB/s at 70 %; the
// same with 32x32x2 MFMAs and with reads one step later).  Tiles of 128 x 64, two a compute unit, ask for three quarters of it and fill the chip
// worse: 1024 rows, 5632 of 1024 107 us against 100; two groups of wavefronts that share a tile's slices 114.
template <bool XS, bool YS>
__global__ void __launch_bounds__(256, 3) gemm_f32_kernel(const GemmF32 g, int tiles_r, int tiles_c) {
  constexpr uint32_t SIDE = 8192, STAGE = 2 * SIDE, STAGES = 3;
  constexpr int CPW = 4;                                          // copies of a wavefront a slice
  __shared__ __attribute__((aligned(1024))) char sAll[STAGES * STAGE];
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;
  const int tid = threadIdx.x, lane = tid & 63, wq = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tr, tc;
  gg_tile_of(gg_xcd_chunk(blockIdx.x, tiles_r * tiles_c), tiles_r, tiles_c, tr, tc);
  const int64_t r0 = (int64_t)tr * 64, c0 = (int64_t)tc * 64;
  const F32Side<XS> X(g.x, r0, g.rows, g.k, wq, lane);
  const F32Side<YS> Y(g.y, c0, g.cols, g.k, wq, lane);
  const int wr = (wq & 1) * 32, wc = (wq >> 1) * 32;
  const F32Reads<XS> RX(wr, lane);
  const F32Reads<YS> RY(wc, lane);
  const int nsl = (int)((g.k + 31) / 32);
  const uint32_t dst = lds0 + 1024u * wq;

  floatx4 acc[2][2], y[2], x[2];                                  // [row block][column block]
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q >> 1][q & 1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < (int)STAGES; ++s) {
    const int4v rx = X.slice(s, nsl), ry = Y.slice(s, nsl);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      copy_1k(X.lane_off, rx, X.off[q], dst + s * STAGE + 4096u * q);
      copy_1k(Y.lane_off, ry, Y.off[q], dst + s * STAGE + SIDE + 4096u * q);
    }
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(2 * CPW) : "memory");
  uint32_t now = 0;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    y[b] = RY.get(lds0 + SIDE, b, 0);
    x[b] = RX.get(lds0, b, 0);
  }
  for (int it = 0; it < nsl; ++it) {
    const uint32_t next = now + STAGE == STAGES * STAGE ? 0 : now + STAGE;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      floatx4 y1[2], x1[2];
      int4v rx, ry;
      if (j == 1) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(CPW) : "memory");
        rx = X.slice(it + 3, nsl);       // (past the end: zeros that nobody uses)
        ry = Y.slice(it + 3, nsl);
      }
      const uint32_t from = lds0 + (j == 1 ? next : now);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          acc[q >> 1][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[q & 1][i], x[q >> 1][i], acc[q >> 1][q & 1], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (i < 2) {
          y1[i] = RY.get(from + SIDE, i, 1 - j);
          x1[i] = RX.get(from, i, 1 - j);
        } else if (j == 1) {
          copy_1k(X.lane_off, rx, X.off[i - 2], dst + now + 4096u * (i - 2));
          copy_1k(Y.lane_off, ry, Y.off[i - 2], dst + now + SIDE + 4096u * (i - 2));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) y[b] = y1[b], x[b] = x1[b];
    }
    now = next;
  }
  // lane (r, g): row r of a block, columns 4 g ..
  const int r = lane & 15, gl = lane >> 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t row = r0 + wr + 16 * (q >> 1) + r, col = c0 + wc + 16 * (q & 1) + 4 * gl;
    if (row >= g.rows || col >= g.cols) continue;      // (cols is a multiple of 4)
    float *dp = g.d + row * g.cols + col;
    floatx4 v = acc[q >> 1][q & 1];
    if (g.accumulate) v += *reinterpret_cast<const floatx4 *>(dp);
    *reinterpret_cast<floatx4 *>(dp) = v;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // no copy outlives the workgroup's LDS
}

template <bool XS, bool YS>
static int launch_f32(const GemmF32 &g, hipStream_t st) {
  const int64_t tr = cdiv(g.rows, 64), tc = cdiv(g.cols, 64);
  hipLaunchKernelGGL((gemm_f32_kernel<XS, YS>), dim3((unsigned)(tr * tc)), dim3(256), 0, st, g, (int)tr, (int)tc);
  DH_LAUNCH_CHECK();
  return DH_OK;
}

// What the kernel takes: 16-byte copies (whole chunks along the contiguous dimensions), offsets of a tile's slice below 2^31 bytes.
static bool gemm_f32_takes(const GemmF32 &g) {
  constexpr int64_t LD = 1 << 20;
  if (!(aligned16(g.x) && aligned16(g.y) && aligned16(g.d)) || g.cols % 4 || (g.x_strided && !g.y_strided)) return false;
  if (!(g.x_strided && g.y_strided) && (g.k % 32 || g.k > LD)) return false;
  return (!g.x_strided || (g.rows % 4 == 0 && g.rows <= LD)) && (!g.y_strided || g.cols <= LD);
}

// Where it is the faster one: its tiles fill five sixths or more of the places of one round of 768 (three a compute unit) or of two, and the
// reduction is short enough that the library's larger tiles have not made up for leaving compute units idle.  us, library / here:
// 1024 rows, 5632 of 1024 (1408 tiles) 110 / 100, 2816 of 1024 (704) 69 / 53, 3072 (768) 55 / 54, data gradients [1024, 1024] x [1024,
// 2816] 70 / 53, [1000, 256] x [256, 5568] (1392) 81 / 31, weight gradients 5632 x 1024 of 1024 rows 117 / 104, 1024 x 2816 70 / 54; but fewer
// tiles, 1024 rows 1536 of 1024 (384) 32 / 37, 777 rows 2816 (572, 0.74 of the places) 45 / 54, a longer reduction 1024 rows, 4000 of
// 2048 (1008, 0.66) 123 / 170, more tiles 1024 rows, 16032 of 1024 (4016) 262 / 300, weight gradients of two rounds from 1281 rows on 3520 x
// 1684 of 1504 rows 137 / 148.  350 random calls within the rule but for these, library / here on average: forwards 1.17, data gradients 1.16, weight gradients
// 1.29; 9 of them below 0.97, the worst 0.90.
// Weight gradients of few rows are launches more than products: up to 192 rows 1.5 times (80 calls, one 0.96), 64 rows 512 x 512 11 / 5; at 227
// rows 4352 x 768 21 / 24.
// The sums run along k in one chain, as the library's do in these ranges: errors against 64 bits are the same (5.7e-7 at k = 1024).
bool gemm_f32_pays(const GemmF32 &g) {
  if (!gemm_f32_takes(g)) return false;
  const int64_t tiles = cdiv(g.rows, 64) * cdiv(g.cols, 64);
  if (tiles > 1536) return false;
  if (g.x_strided && g.k <= 192) return true;
  return g.k <= (!g.x_strided ? 1024 : tiles > 768 ? 1280 : 1536) && tiles >= 640 && 6 * tiles >= 5 * 768 * cdiv(tiles, 768);
}

int launch_gemm_f32(const GemmF32 &g, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  if (g.x_strided) return launch_f32<true, true>(g, st);
  return g.y_strided ? launch_f32<false, true>(g, st) : launch_f32<false, false>(g, st);
}

}  // namespace dh
