// Grouped GEMM on gfx950 MFMA (bf16/fp16 inputs, fp32 accumulate) for one
// expert-parallel rank: every local expert multiplies its own contiguous block
// of permuted rows.
//
// One template covers the three products a SwiGLU expert needs:
//   NT  c[r, n]  = sum_k a[r, k] * w[g][n, k]      forward  (both k-contiguous)
//   NN  c[r, n]  = sum_k a[r, k] * w[g][k, n]      dgrad    (w strided in k)
//   TN  c[g][m,n] = sum_r a[r, m] * b[r, n]        wgrad    (both strided in k = r)
// Two kernels.  grouped_gemm_w8_kernel (products that fill the chip): a workgroup per 256x256 tile, eight wavefronts in two
// alternating groups; with a workspace further workgroups of the launch may take the last round of tiles in k pieces.
// grouped_gemm_t_kernel (everything else): smaller tiles, copied straight to LDS, split along k where
// there are few of them.  k-contiguous operands are read from LDS as 16-byte row fragments; k-strided operands stay
// row-major in LDS and are read with transpose loads, so no operand is ever transposed in memory.
// The product is formed as C^T (weights in the MFMA A slot) so that each lane
// ends up with runs of 4 consecutive output columns of one row: 8-byte stores.
// Group row ranges are read on the device from the offsets table.
#include <cmath>

#include "mma.h"
#include "tile_order.h"
#include <atomic>

namespace dh {

constexpr int GG_MAX_GROUPS = 64;

struct GGParams {
  const void *a, *b;
  void *c;
  const int32_t *offs;
  int groups;
  int64_t m_dim;   // TN: columns of a (= rows of c[g]); NT/NN: unused
  int64_t n_dim;   // output columns
  int64_t k_dim;   // NT/NN: reduction length; TN: unused (comes from offs)
  int64_t lda, ldb, ldc;
  int64_t b_group_stride, c_group_stride;
  int tiles_m, tiles_n;  // grid extents (tiles_m is an upper bound for NT/NN)
  int accumulate;
  int max_rows;          // rows the stacked operands hold: group ranges read from offs are cut off there
  float *ws;             // split last round: fp32 partial tiles, one per workgroup
  int zero_tail;         // NT/NN on grouped_gemm_w8_kernel: the kernel itself zeroes the rows of c past the last group
  int sk_grid;           // grouped_gemm_w8_kernel: > 0: so many workgroups behind the tiles may take the last round of them in pieces;
                         // grouped_gemm_t_kernel, NT/NN: > 0: places for workgroups, over which the tiles may be split along k
  int pieces;            // grouped_gemm_t_kernel, TN: k pieces per tile
};

// Entry i of the offsets table; without a table there is one group of all max_rows rows.
__device__ __forceinline__ int gg_off(const GGParams &p, int i) { return p.offs ? p.offs[i] : i * p.max_rows; }

// A group's row range as the kernels use it: relative to the first group and never past the rows the caller's
// buffers hold, whatever the offsets say (they live on the device, so the host cannot check them).
__device__ __forceinline__ int gg_clamp_row(int r, int max_rows) { return r < 0 ? 0 : (r > max_rows ? max_rows : r); }

// The groups' row ranges held one group per lane (at most 64 groups), read with ONE vector load per wavefront
// instead of a chain of scalar loads per group (0.25 us per group and tile): lane g has group g's clamped range
// and the inclusive prefix sum of the groups' tile counts (tiles of BM rows).  Call with all lanes active.
struct GGGroupTable { int rb, re, incl; };
template <int BM = 256>
__device__ __forceinline__ GGGroupTable gg_group_table(const GGParams &p, int base, int &tiles_m) {
  const int lane = threadIdx.x & 63;
  int rb = 0, re = 0;
  if (lane < p.groups) {
    rb = gg_clamp_row(gg_off(p, lane) - base, p.max_rows);
    re = gg_clamp_row(gg_off(p, lane + 1) - base, p.max_rows);
  }
  int incl = (re - rb + BM - 1) / BM;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  tiles_m = __builtin_amdgcn_readlane(incl, 63);
  return GGGroupTable{rb, re, incl};
}
// The group that holds m tile tm_all (< tiles_m) of the stacked rows, its row range and the tile's index inside it.
template <int BM = 256>
__device__ __forceinline__ void gg_locate(const GGGroupTable &gt, int tm_all, int &g, int &rb, int &re, int &tm) {
  g = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(gt.incl > tm_all)));
  rb = __builtin_amdgcn_readlane(gt.rb, g);
  re = __builtin_amdgcn_readlane(gt.re, g);
  tm = tm_all - (__builtin_amdgcn_readlane(gt.incl, g) - (re - rb + BM - 1) / BM);
}

// ---- 256x256 tiles, eight wavefronts in two alternating groups ---------------------------------------------------
// Eight wavefronts of 128x64 outputs (two per SIMD) on v_mfma_f32_16x16x32: under a sustained load this board is bound by
// power, and that instruction delivers 2.03 PFLOP/s where 32x32x16 stops at 1.79 (loops of nothing else on normal data).
// The operands of a 64-deep k slice are copied straight to LDS (two stages of four 16 KB regions: the A rows and the B
// columns of the tile in two halves each), and every wavefront works through a slice in four quarters of its outputs, a
// quarter being [reads of fragments, copies | 16 MFMAs, more reads among them], each half of it ended by a barrier.  The
// wavefronts 4..7 start one barrier late, so that on every SIMD one wavefront has its 16 MFMAs while the other reads LDS and
// issues copies.  Slice s, F = the half of B that is multiplied first (s % 2), G = the other:
//   cluster 0  read G                             1  A0 x F, read A1
//           2  read A1     copy A0 of s + 2       3  A0 x G, read A1
//           4  read A0'    copy F of s + 2        5  A1 x G, read A0'      (A0', F': of slice s + 1)
//           6  read F'     copy G, A1 of s + 2    7  A1 x F, read A0'
// Fragments are read at least one cluster of MFMAs ahead of their use.  Why no copy overtakes a read: a read cluster begins
// with the wait for the wavefront's earlier reads, so what was read up to cluster c is in registers, for the leading group by
// cluster c + 2 and for the other one barrier later; the copies into a region go out behind the next barrier after that.
// Why no read overtakes a copy: two clusters before a region is read every wavefront waits for its own copies of it (copies
// complete in order, so `vmcnt` counts those issued behind them); both groups are past that wait when the leading one
// reads.  8 copies stay in flight across every barrier.
//
// LDS regions: a k-contiguous operand as [128 rows][64 k] (128-byte rows, 16-byte chunk XOR (row / 2) % 8: row-fragment reads
// hit 16 different chunks), a k-strided one as [64 k][128 columns] (256-byte rows, chunk XOR 4 (k % 4) + (k / 4) % 4), read as
// fragments by LDS transpose reads.  The XOR is applied to the global chunk that a lane fetches.  Buffer descriptors do the edge
// handling: their length is cut at the group's (or n's) last row, so that rows past the end read as zero and no access leaves
// the operands, whatever the offsets table says; slices past the last one are copied with a length of zero, or the old
// tile is copied in their place (below).
// us, against the kernel before it (four wavefronts on 32x32x16, operands staged through registers); two groups of 2048 rows:
// NT n = 28672 of 4096 764 -> 705, n = 4096 of 14336 375 -> 331; NN 778 -> 704 and 380 -> 336; TN 862 -> 778 and 425 -> 389,
// accumulating 1091 -> 806 and 531 -> 413.  One group of 8192 x 8192 x 8192: NT 802 -> 721 (1.52 PFLOP/s; the library 709), TN
// 849 -> 783 (1.40; the library 928).  What bounds it: power (matrix pipes 82 % busy at 1.76 GHz, TN 71 % at 1.92), and per tile
// about 8 us of first copies and last stores.
// The outputs of a wavefront (wm = w / 4, wn = w % 4): quarter (qm, qn) holds rows 128 qm + 64 wm + 16 mi + .. and columns
// 128 qn + 32 wn + 16 nj + .. of the tile; its 16x16 blocks lie transposed in the accumulators (lane % 16: output row, four
// consecutive columns 4 (lane / 16) + .. a lane).
typedef floatx4 GGAcc8[2][2][4][2];          // [qm][qn][mi][nj]

// Stores a tile through LDS ([256][512 bytes], the 16-byte chunk index XORed with row % 16: 8-byte accesses of 16 rows fall on
// different banks), so that 32 lanes write a row of 512 bytes.  ADD: LDS holds the old tile, to which each lane adds what it
// holds, with one rounding.
template <typename T, bool ADD>
__device__ __forceinline__ void gg_w8_store(const GGAcc8 &acc, unsigned char *smem, const GGParams &p, T *cbase, int m0, int n0,
                                            int a_rext, int b_rext) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 2, wn = w & 3;
  struct alignas(8) Q4 { T v[4]; };
  const int r16 = lane & 15, g4 = lane >> 4;
  unsigned char *mine = smem + (64 * wm + r16) * 512 + (g4 & 1) * 8;
  const int ch = (4 * wn + (g4 >> 1)) ^ r16;                      // chunk of columns 32 wn + 4 g4; + 16 columns: two chunks on
#pragma unroll
  for (int qm = 0; qm < 2; ++qm)
#pragma unroll
    for (int qn = 0; qn < 2; ++qn)
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int nj = 0; nj < 2; ++nj) {
          Q4 *dst = reinterpret_cast<Q4 *>(mine + (128 * qm + 16 * mi) * 512 + ((ch ^ (2 * nj)) + 16 * qn) * 16);
          const floatx4 av = acc[qm][qn][mi][nj];
          Q4 o;
          if constexpr (ADD) {
            const Q4 old = *dst;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(av[e] + static_cast<float>(old.v[e]));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(av[e]);
          }
          *dst = o;
        }
  __syncthreads();
  const int er = tid >> 5, ec = tid & 31;                         // row of 16 and chunk
  const unsigned char *src = smem + er * 512 + ((ec ^ er) << 4);
  T *row0 = cbase + (int64_t)(m0 + er) * p.ldc + n0 + 8 * ec;
  if (8 * ec < b_rext) {
#pragma unroll 8
    for (int it = 0; it < 16; ++it)
      if (16 * it + er < a_rext)
        *reinterpret_cast<dh_u32x4 *>(row0 + (int64_t)(16 * it) * p.ldc) = *reinterpret_cast<const dh_u32x4 *>(src + it * (16 * 512));
  }
}

// k pieces per tile of the last round: as many as there are workgroups per tile, each at least one slice.
__device__ __forceinline__ int gg_sk_pieces(int grid, int rem, int nsl) {
  if (rem <= 0) return 1;
  const int pc = grid / rem;
  return pc < 1 ? 1 : (pc > nsl ? (nsl > 0 ? nsl : 1) : pc);
}

// FORM 0: NT (both operands k-contiguous); 1: NN (b k-strided); 2: TN (both k-strided, k = the group's rows, one output
// per group).
template <typename T, int FORM, bool SK>
__global__ void __launch_bounds__(512) grouped_gemm_w8_kernel(const GGParams p) {
  constexpr bool BKS = FORM >= 1, AKS = FORM == 2;
  static_assert(!(AKS && SK), "the wgrad form has many tiles and a short k: it is never split");
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int BM = 256;
  constexpr uint32_t REG = 16384, STAGEB = 4 * REG, OFF_B = 2 * REG;     // regions A0 A1 B0 B1
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * STAGEB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w >> 2, wn = w & 3;
  const int c = lane & 15, g4 = lane >> 4;
  const int nsl = (int)((p.k_dim + 63) / 64);
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const uint32_t lda_b = (uint32_t)p.lda * (uint32_t)sizeof(T), ldb_b = (uint32_t)p.ldb * (uint32_t)sizeof(T);
  const int base = gg_off(p, 0);

  // Rows of c past the last group, up to max_rows (usually none): zeroed here, a row per workgroup at a time, instead
  // of by a kernel of its own in front of this one (5 us per product).
  if constexpr (!AKS) {
    if (p.zero_tail) {
      const int first = gg_clamp_row(gg_off(p, p.groups) - base, p.max_rows);
      const int nv = (int)(p.n_dim / 8);
      for (int r = first + (int)blockIdx.x; r < p.max_rows; r += (int)gridDim.x) {
        T *row = reinterpret_cast<T *>(p.c) + (int64_t)r * p.ldc;
        for (int v = tid; v < nv; v += 512) *reinterpret_cast<dh_u32x4 *>(row + 8 * v) = dh_u32x4{0u, 0u, 0u, 0u};
      }
    }
  }

  // ---- copies: a region is 16 blocks of 1 KB, a wavefront takes blocks 2 w and 2 w + 1.  k-contiguous: a block is 8 rows (a lane:
  // row lane / 8, chunk lane % 8); k-strided: 4 k rows (row lane / 16, chunk lane % 16)
  uint32_t va[2], vb[2];                                                 // lane offsets of the two blocks
  {
    const int r8 = lane >> 3, ch = (lane & 7) ^ (r8 >> 1), r4 = lane >> 4, cs = (lane & 15) ^ (4 * r4);
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int b = 2 * w + x;
      const uint32_t kc = (uint32_t)((ch ^ (4 * x)) << 4), ks = (uint32_t)((cs ^ (b & 3)) << 4);
      va[x] = AKS ? (uint32_t)(4 * b + r4) * lda_b + ks : (uint32_t)(8 * b + r8) * lda_b + kc;
      vb[x] = BKS ? (uint32_t)(4 * b + r4) * ldb_b + ks : (uint32_t)(8 * b + r8) * ldb_b + kc;
    }
  }
  const uint32_t kstep_a = AKS ? 64 * lda_b : 128, kstep_b = BKS ? 64 * ldb_b : 128;        // bytes from one k slice to the next
  const uint32_t half_a = AKS ? 256 : 128 * lda_b, half_b = BKS ? 256 : 128 * ldb_b;        // bytes to the second half of the tile
  const uint32_t cp_lds = lds0 + (uint32_t)(w * 2048);

  // ---- fragments: lane row (column) c of a 16-row block, k = 8 g4 + 0..7 of a step of 32
  const uint32_t sw = (uint32_t)((g4 ^ ((c >> 1) & 7)) << 4);
  const uint32_t fa_lane = (uint32_t)((wm * 64 + c) * 128) + sw, fb_lane = (uint32_t)((wn * 32 + c) * 128) + sw;   // step: XOR 64; block: + 2048
  const int tx = 4 * (c >> 2) + ((2 * g4) & 3);
  const uint32_t t_row = (uint32_t)((8 * g4 + (c >> 2)) * 256 + (c & 1) * 8);
  const uint32_t t_lo = t_row + (uint32_t)((((c & 3) >> 1) ^ tx) << 4);                    // k rows 8 g4 + 0..3 of a step
  const uint32_t t_hi = t_row + 1024 + (uint32_t)((((c & 3) >> 1) ^ (tx + 1)) << 4);       // k rows 8 g4 + 4..7
  typedef __attribute__((address_space(3))) const Frag *lds_frag;
  typedef short4v __attribute__((address_space(3))) *lds_tr;
  auto tr_frag = [&](uint32_t region, int blk, int ks) {                 // 16 columns `blk` of a k-strided region
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(region + (t_lo ^ (uint32_t)(blk << 5)) + (uint32_t)(ks * 8192)));
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(region + (t_hi ^ (uint32_t)(blk << 5)) + (uint32_t)(ks * 8192)));
    return frag_join<T>(lo, hi);
  };
  auto frag_a = [&](uint32_t region, int mi, int ks) -> Frag {
    if constexpr (AKS) return tr_frag(region, wm * 4 + mi, ks);
    else return *(lds_frag)(region + (fa_lane ^ (uint32_t)(ks << 6)) + (uint32_t)(mi * 2048));
  };
  auto frag_b = [&](uint32_t region, int nj, int ks) -> Frag {
    if constexpr (BKS) return tr_frag(region, wn * 2 + nj, ks);
    else return *(lds_frag)(region + (fb_lane ^ (uint32_t)(ks << 6)) + (uint32_t)(nj * 2048));
  };

  // One segment: slices [s0, s1) of the tile (g, tm, tn).  part == nullptr: the segment is the whole k range and the
  // result goes to c; else the fp32 partial sums go to part (accumulator layout: 1 KB per wavefront instruction;
  // gg_split_reduce_kernel sums the pieces of a tile in k order).
  auto segment = [&](int g, int row_begin, int row_end, int tm, int tn, int s0, int s1, float *part) {
    // NT / NN: output rows m0.. of the stacked rows; TN: output rows m0.. of group g's own [m_dim, n_dim] result
    const int n0 = tn * 256, m0 = AKS ? tm * BM : row_begin + tm * BM;
    const int a_rext = AKS ? (int)(p.m_dim - m0) : row_end - m0, b_rext = (int)(p.n_dim - n0);
    const T *ag = reinterpret_cast<const T *>(p.a) + (AKS ? (int64_t)row_begin * p.lda + m0 : (int64_t)m0 * p.lda);
    const T *bg = AKS ? reinterpret_cast<const T *>(p.b) + (int64_t)row_begin * p.ldb + n0
                      : reinterpret_cast<const T *>(p.b) + (int64_t)g * p.b_group_stride + (BKS ? (int64_t)n0 : (int64_t)n0 * p.ldb);
    // One descriptor per operand, cut at the last row of the group (of n): the hardware compares the lane offset plus
    // the scalar offset with the length, so a row past the end reads as zero whichever block it is in.
    // (k-strided operands: cut at the last k row, i.e. the group's last row for TN; in the other direction a tile that
    // reaches past n or m reads what follows in the operand, into outputs that are not stored)
    const int4v rsa_ = AKS ? raw_rsrc(ag, (int64_t)(row_end - row_begin) * lda_b - (int64_t)m0 * (int)sizeof(T))
                             : raw_rsrc(ag, (int64_t)(a_rext < 256 ? a_rext : 256) * lda_b);
    const int4v rsb_ = AKS ? raw_rsrc(bg, (int64_t)(row_end - row_begin) * ldb_b - (int64_t)n0 * (int)sizeof(T))
                       : BKS ? raw_rsrc(bg, (int64_t)p.k_dim * ldb_b - (int64_t)n0 * (int)sizeof(T))
                             : raw_rsrc(bg, (int64_t)(b_rext < 256 ? b_rext : 256) * ldb_b);
    // The descriptors come out of v_readfirstlane, and a memory instruction may read such a scalar register five wait
    // states later at the earliest.  The compiler keeps that distance for its own instructions, not for the copies issued
    // from assembly: without this the first of them went out with the previous contents of the length, now and then
    // (a group of fewer than 64 rows then took rows of its neighbour into its weight gradient).
    int4v rsa = rsa_, rsb = rsb_;
    asm volatile("s_nop 4" : "+s"(rsa), "+s"(rsb));
    const int cnt = s1 - s0;                                             // slices of this segment
    // TN: what is added to (nothing to read if nothing is)
    const uint32_t ldc_b = (uint32_t)p.ldc * (uint32_t)sizeof(T);
    T *const cbase = reinterpret_cast<T *>(p.c) + (AKS ? (int64_t)g * p.c_group_stride : 0);
    int4v rsc = AKS ? raw_rsrc(cbase + (int64_t)m0 * p.ldc + n0,
                                 p.accumulate ? (int64_t)(a_rext < 256 ? a_rext : 256) * ldc_b - (int64_t)n0 * (int)sizeof(T) : 0)
                       : int4v{0, 0, 0, 0};
    if constexpr (AKS) asm volatile("s_nop 4" : "+s"(rsc));
    // What the copies of a slice read.  For the slices past the last one it is switched to nothing, or, for TN, to the old tile: rows
    // of 512 bytes one behind the other over both stages, which are full of it when the last MFMAs end (a read of its own
    // behind them took 5 us a tile).
    uint32_t ca[2] = {va[0], va[1]}, cb[2] = {vb[0], vb[1]};
    bool past = false;
    auto past_the_last = [&] {
      past = true;
      if constexpr (AKS) {
        rsa = rsb = rsc;
#pragma unroll
        for (int x = 0; x < 2; ++x)
          ca[x] = cb[x] = (uint32_t)(2 * (2 * w + x) + (lane >> 5)) * ldc_b + (uint32_t)(((lane & 31) ^ (((4 * w + 2 * x) & 15) | (lane >> 5))) << 4);
      } else {
        rsa[2] = rsb[2] = 0;
      }
    };
    // a last slice of k_dim % 64: a k-contiguous operand's chunks past it read as zero (a k-strided one is cut by its descriptor)
    const int tail = AKS ? 0 : (int)(p.k_dim % 64);
    auto the_last = [&] {
      const int ch = (lane & 7) ^ (lane >> 4);                           // global chunk of the lane's copies: XOR 4 for the second
#pragma unroll
      for (int x = 0; x < 2; ++x)
        if ((ch ^ (4 * x)) * 8 >= tail) {
          ca[x] = 0x80000000u;                                           // past any descriptor's end
          if constexpr (!BKS) cb[x] = 0x80000000u;
        }
    };
    // before the copies of slice s (of this segment)
    auto turn_to = [&](int s) {
      if (s >= cnt) past_the_last();
      else if (!AKS && tail != 0 && s0 + s == nsl - 1) the_last();
    };
    // half `h` of an operand's slice s (of this segment) into stage `stage`
    auto copy_a = [&](int h, int s, uint32_t stage) {
      const uint32_t at = stage + (uint32_t)h * REG;
      const uint32_t off = AKS && past ? at / 512 * ldc_b : (uint32_t)(s0 + s) * kstep_a + (uint32_t)h * half_a;
#pragma unroll
      for (int x = 0; x < 2; ++x) copy_1k(ca[x], rsa, off, cp_lds + at + (uint32_t)(x * 1024));
    };
    auto copy_b = [&](int h, int s, uint32_t stage) {
      const uint32_t at = stage + OFF_B + (uint32_t)h * REG;
      const uint32_t off = AKS && past ? at / 512 * ldc_b : (uint32_t)(s0 + s) * kstep_b + (uint32_t)h * half_b;
#pragma unroll
      for (int x = 0; x < 2; ++x) copy_1k(cb[x], rsb, off, cp_lds + at + (uint32_t)(x * 1024));
    };
    GGAcc8 acc;
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i >> 4][(i >> 3) & 1][(i >> 1) & 3][i & 1] = floatx4{0.f, 0.f, 0.f, 0.f};
    Frag fa[2][4][2], fb[2][2][2];                                       // [half][block][step]
    // 16 MFMAs; behind every second one a fragment read of what `rd(x)` says
    auto mma_quarter = [&](int qm, int qn, auto rd) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int ks = x >> 3, mi = (x >> 1) & 3, nj = x & 1;
        acc[qm][qn][mi][nj] = M::mma16(fb[qn][nj][ks], fa[qm][mi][ks], acc[qm][qn][mi][nj]);   // C^T: lane column = output row
        if (x & 1) {
          __builtin_amdgcn_sched_barrier(0);
          rd(x >> 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
    };
    auto read_a = [&](int h, uint32_t region, int x0, int x1) {          // fragments x0..x1 of the half's eight
#pragma unroll
      for (int x = x0; x < x1; ++x) fa[h][x & 3][x >> 2] = frag_a(region, x & 3, x >> 2);
    };
    auto read_b = [&](int h, uint32_t region) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int nj = 0; nj < 2; ++nj) fb[h][nj][ks] = frag_b(region, nj, ks);
    };
#define GG_W8_BARRIER()                       \
    do {                                      \
      __builtin_amdgcn_sched_barrier(0);      \
      asm volatile("s_barrier" ::: "memory"); \
      __builtin_amdgcn_sched_barrier(0);      \
    } while (0)
#define GG_W8_READS_DONE() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
#define GG_W8_WAIT_BARRIER(n)                                           \
    do {                                                                \
      __builtin_amdgcn_sched_barrier(0);                                \
      asm volatile("s_waitcnt vmcnt(" #n ")\n\ts_barrier" ::: "memory"); \
      __builtin_amdgcn_sched_barrier(0);                                \
    } while (0)

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                    // (the zeroed rows' stores are not part of the counts below)
    turn_to(0);
    copy_a(0, 0, 0); copy_b(0, 0, 0); copy_b(1, 0, 0); copy_a(1, 0, 0);
    turn_to(1);
    copy_a(0, 1, STAGEB); copy_b(1, 1, STAGEB); copy_b(0, 1, STAGEB); copy_a(1, 1, STAGEB);
    GG_W8_WAIT_BARRIER(8);
    if (w >= 4) GG_W8_BARRIER();
    read_a(0, lds0, 0, 8);
    read_b(0, lds0 + OFF_B);
    uint32_t cur = 0;
    auto slice = [&](auto fc, int s) {
      constexpr int F = decltype(fc)::value, G = F ^ 1;                  // the half of B that is multiplied first (s % 2), and the other
      const uint32_t nxt = cur ^ STAGEB, sa = lds0 + cur, sb = sa + OFF_B, na = lds0 + nxt, nb = na + OFF_B;
      turn_to(s + 2);
      GG_W8_READS_DONE();
      read_b(G, sb + G * REG);
      GG_W8_BARRIER();
      mma_quarter(0, F, [&](int x) { if (x < 3) read_a(1, sa + REG, x, x + 1); });
      GG_W8_BARRIER();
      GG_W8_READS_DONE();
      read_a(1, sa + REG, 3, 6);
      copy_a(0, s + 2, cur);
      GG_W8_WAIT_BARRIER(8);
      mma_quarter(0, G, [&](int x) { if (x < 2) read_a(1, sa + REG, 6 + x, 7 + x); });
      GG_W8_BARRIER();
      GG_W8_READS_DONE();
      read_a(0, na, 0, 3);
      copy_b(F, s + 2, cur);
      GG_W8_WAIT_BARRIER(8);
      mma_quarter(1, G, [&](int x) { if (x < 3) read_a(0, na, 3 + x, 4 + x); });
      GG_W8_BARRIER();
      GG_W8_READS_DONE();
      read_b(G, nb + G * REG);
      copy_b(G, s + 2, cur);
      copy_a(1, s + 2, cur);
      GG_W8_WAIT_BARRIER(8);
      mma_quarter(1, F, [&](int x) { if (x < 2) read_a(0, na, 6 + x, 7 + x); });
      GG_W8_BARRIER();
      cur = nxt;
    };
    int s = 0;
#pragma unroll 1
    for (; s + 1 < cnt; s += 2) {
      slice(std::integral_constant<int, 0>{}, s);
      slice(std::integral_constant<int, 1>{}, s + 1);
    }
    if (s < cnt) slice(std::integral_constant<int, 0>{}, s);
    if (w < 4) GG_W8_BARRIER();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                    // the last copies (zeros) have landed before the stages are used again
    __syncthreads();

    if (SK && part != nullptr) {
      // 16 bytes per lane and instruction: piece w * 32 + block of the tile, 1 KB each
      float *dst = part + (size_t)w * 32 * 256 + (size_t)lane * 4;
#pragma unroll
      for (int i = 0; i < 32; ++i) *reinterpret_cast<floatx4 *>(dst + (size_t)i * 256) = acc[i >> 4][(i >> 3) & 1][(i >> 1) & 3][i & 1];
      return;
    }
    if (AKS && p.accumulate) gg_w8_store<T, true>(acc, smem, p, cbase, m0, n0, a_rext, b_rext);
    else gg_w8_store<T, false>(acc, smem, p, cbase, m0, n0, a_rext, b_rext);
  };

  if constexpr (AKS) {
    // one output of tiles_m x tiles_n tiles per group (blockIdx.y); k = the group's rows, the last slice cut there
    const int ntiles = p.tiles_m * p.tiles_n;
    int pid = blockIdx.x;
    pid = gg_xcd_chunk(pid, ntiles);
    const int g = blockIdx.y;
    const int rb = gg_clamp_row(gg_off(p, g) - base, p.max_rows), re = gg_clamp_row(gg_off(p, g + 1) - base, p.max_rows);
    int tm, tn;
    gg_tile_of(pid, p.tiles_m, p.tiles_n, tm, tn);
    segment(g, rb, re, tm, tn, 0, (re - rb + 63) / 64, nullptr);
  } else {
    // The grid is sized for the host's upper bound of the tile count (it does not know how the rows split into
    // groups); the chunks of the XCDs are cut from the real count, so that every XCD gets its share of real tiles.
    int tiles_m;
    const GGGroupTable gt = gg_group_table(p, base, tiles_m);
    const int ntiles = tiles_m * p.tiles_n;
    int kept = ntiles, rem = 0, pieces = 1;
    if constexpr (SK) {
      // The tiles (in the order of gg_tile_of) run in rounds of sk_grid = the number of compute units.  When the last round
      // holds at most half as many tiles as there are compute units it is split along k: as many pieces per tile as fit
      // (unit w behind the full rounds: tile w % rem, piece w / rem, so that neighbours work on neighbouring tiles), summed
      // afterwards in k order.  288 tiles on 256 compute units then take 1 1/8 tile times instead of 2.  The pieces are the last
      // workgroups of the same launch: they start as compute units run out of full-round tiles, not when the last of them has
      // ended.  bf16 NT, 1280 rows x 2 groups, 7168 x 4096: 82.8 -> 78.5 us against a kernel of their own behind; 16 groups of
      // 256 rows, 4096 x 2816: 149 -> 146; nothing to split: one launch of 5 us less.  (A resident workgroup that also looped
      // over the full rounds was 3-6 % slower on them than one workgroup per tile.)
      const int full = ntiles / p.sk_grid;
      rem = ntiles - full * p.sk_grid;
      pieces = gg_sk_pieces(p.sk_grid, rem, nsl);
      if (pieces > 1) kept = full * p.sk_grid;
    }
    int pid, s0 = 0, s1 = nsl;
    float *part = nullptr;
    if ((int)blockIdx.x < kept) {
      pid = gg_xcd_chunk((int)blockIdx.x, kept);                      // (the XCDs share the tiles that are computed here)
    } else if (SK && pieces > 1 && (int)blockIdx.x - kept < p.sk_grid) {
      const int wg = gg_xcd_chunk((int)blockIdx.x - kept, p.sk_grid);  // neighbouring tiles on one XCD (kept: whole rounds)
      if (wg >= rem * pieces) return;
      const int pc = wg / rem;
      pid = kept + wg % rem;
      s0 = pc * nsl / pieces;
      s1 = (pc + 1) * nsl / pieces;
      part = p.ws + (size_t)wg * (256 * 256);
    } else {
      return;
    }
    int tm_all, tn, g, rb, re, tm;
    gg_tile_of(pid, tiles_m, p.tiles_n, tm_all, tn);
    gg_locate(gt, tm_all, g, rb, re, tm);
    segment(g, rb, re, tm, tn, s0, s1, part);
  }
}
#undef GG_W8_BARRIER
#undef GG_W8_WAIT_BARRIER
#undef GG_W8_READS_DONE

// Sums the k pieces of the tiles of a split last round, in k order (deterministic), and stores the tiles.
// 16 workgroups per tile of that round: a wavefront takes four neighbouring 16x16 blocks (two by two) of the accumulator layout,
// reads their 4 KB of every piece (1 KB per instruction) and writes 4 columns per lane and block.
template <typename T>
__global__ void __launch_bounds__(256) gg_split_reduce_kernel(const GGParams p, int sk_grid) {
  constexpr int BM = 256;
  const int nsl = (int)((p.k_dim + 63) / 64);
  const int base = gg_off(p, 0);
  int tiles_m = 0;
  for (int gi = 0; gi < p.groups; ++gi)
    tiles_m += (gg_clamp_row(gg_off(p, gi + 1) - base, p.max_rows) - gg_clamp_row(gg_off(p, gi) - base, p.max_rows) + BM - 1) / BM;
  const int tiles = tiles_m * p.tiles_n, full = tiles / sk_grid, rem = tiles - full * sk_grid;
  const int ts = blockIdx.x / 16;                       // tile of the last round
  if (ts >= rem || nsl == 0) return;
  const int pieces = gg_sk_pieces(sk_grid, rem, nsl);
  if (pieces == 1) return;
  const int t = full * sk_grid + ts;
  const int tid = threadIdx.x, lane = tid & 63;
  const int unit = (blockIdx.x % 16) * 4 + (tid >> 6);  // blocks 4 unit .. 4 unit + 3 of the tile's 256
  const int w = unit >> 3, q = unit & 7;                // wavefront of the tile; (qm, qn, mi / 2)
  floatx4 acc[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int pc = 0; pc < pieces; ++pc) {
    const float *src = p.ws + (size_t)(pc * rem + ts) * (256 * 256) + (size_t)unit * (4 * 256) + (size_t)lane * 4;
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] += *reinterpret_cast<const floatx4 *>(src + x * 256);
  }
  int tm, tn;
  gg_tile_of(t, tiles_m, p.tiles_n, tm, tn);
  int rb = 0, re = 0;
  for (int gi = 0; gi < p.groups; ++gi) {
    rb = gg_clamp_row(gg_off(p, gi) - base, p.max_rows); re = gg_clamp_row(gg_off(p, gi + 1) - base, p.max_rows);
    const int nt = (re - rb + BM - 1) / BM;
    if (tm < nt) break;
    tm -= nt;
  }
  const int m = rb + tm * BM + 128 * (q >> 2) + 64 * (w >> 2) + 32 * (q & 1) + (lane & 15);         // + 16 (x / 2)
  const int n = tn * 256 + 128 * ((q >> 1) & 1) + 32 * (w & 3) + 4 * (lane >> 4);                   // + 16 (x % 2)
  struct alignas(8) Q4 { T v[4]; };
#pragma unroll
  for (int x = 0; x < 4; ++x)
    if (m + 16 * (x >> 1) < re && n + 16 * (x & 1) < p.n_dim) {
      Q4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[x][e]);
      *reinterpret_cast<Q4 *>(reinterpret_cast<T *>(p.c) + (int64_t)(m + 16 * (x >> 1)) * p.ldc + n + 16 * (x & 1)) = o;
    }
}

// ---- smaller tiles, two workgroups per compute unit ---------------------------------------------------------
// Everything that does not fill the chip with 256x256 tiles, and weight gradients of groups of few rows.  What bounds
// these: weights that are read once for a handful of rows (HBM), reductions that leave most of the chip idle, and fixed
// costs (first loads, last stores) that one workgroup per compute unit cannot hide.  So: BM x 128 tiles with BM = 32, 64
// or 128 by the rows a group has, four wavefronts, operands copied straight to LDS (no staging registers), two
// workgroups per compute unit so that one computes while the other loads or stores, and the reduction split over
// workgroups (fp32 pieces, summed in k order by gg_t_reduce_kernel) when there are fewer tiles than places for them.
// An expert FFN of 2000 rows in 8 groups (hidden 1024, ffn 2816), us per product against a register-staged 128x128 kernel
// with one workgroup per compute unit: fc1 52 -> 41, fc2 45 -> 29, their data gradients 30 -> 22 and 85 -> 42, weight
// gradients 32 -> 26 and 53 -> 44; 53 rows (hidden 2048, ffn 3584): 42 -> 37 (6.3 TB/s of weights), 51 -> 25, 35 -> 25,
// 102 -> 42.  In the steady state two workgroups of a compute unit take 0.95 us per slice of two 128x128 tiles
// (1.13 PFLOP/s, 27 bytes per cycle and compute unit out of L2); the start and end of a round of tiles cost 5 us.
//
// With more 128x128 tiles than that, a single stage and four workgroups a compute unit (34 KB of LDS, at most 128 registers) hide
// loads and stores behind each other better than two of two stages: a workgroup waits for each of its slices, three others
// work meanwhile.  Weight gradients of few rows, mostly stores: 16 experts of 72 rows, 5632 x 4096 236 -> 180 us (3.1 -> 4.1 TB/s),
// 2816 x 4096 118 -> 96; 8 x 250 rows, 5632 x 1024 44 -> 38, 1024 rows 107 -> 95.
//
// LDS: a k-contiguous operand as [rows][64 k] (128-byte rows, 16-byte chunk XOR (row / 2) % 8), a k-strided one as
// [64 k][128 columns] (256-byte rows, chunk XOR 4 (k % 4) + (k / 4) % 4), as in grouped_gemm_w8_kernel; a wavefront
// copies 1 KB per instruction, so the XOR is applied to the global chunk that a lane fetches.  Buffer descriptors cut
// the operands at the group's last row (k-strided: last k row), past which a copy writes zeros; columns past n read
// what follows in the same operand and end in outputs that are not stored.
constexpr int64_t GG_MAX_LD = (1 << 22) - 8;       // row lengths (elements) of the tiled kernels: 256 rows stay inside 31-bit byte offsets

// k pieces per tile: what fills the chip's places, each at least 8 slices long (a piece costs about as much traffic for
// its fp32 tile, written and read, as four slices of operands).
__host__ __device__ __forceinline__ int gg_t_pieces(int slots, int tiles, int nsl) {
  if (tiles <= 0 || 2 * tiles > slots) return 1;
  int pc = slots / tiles;
  if (pc > nsl / 8) pc = nsl / 8;
  if (pc > 16) pc = 16;
  return pc < 2 || nsl - nsl / pc < 12 ? 1 : pc;
}

template <int FORM, int BM, int BN, int ST = 0> struct GGT {
  static constexpr bool AKS = FORM == 2, BKS = FORM >= 1;
  static constexpr int NW = BN / 32;                            // wavefronts
  static constexpr int WM = BM == 32 ? 1 : 2, WN = NW / WM;     // over the tile
  static constexpr int MI = BM / (32 * WM), NI = BN / (32 * WN); // 32x32 blocks of a wavefront
  static constexpr int NST = ST ? ST : BN == 256 ? 3 : BM == 128 ? 2 : BM == 64 ? 3 : 4;  // stages: 144 KB; 64, 72, 80 KB
  static constexpr int ABYTES = BM * 128, STAGE = ABYTES + BN * 128;
  static constexpr int ACPW = BM / (8 * NW), BCPW = BN / (8 * NW), CPW = ACPW + BCPW;   // copies of a wavefront per slice
  static constexpr int PER_CU = ST == 1 ? 4 : BN == 256 ? 1 : 2; // workgroups that share a compute unit
  static constexpr int EP = NI * 64 + 8, EPB = NW * 32 * MI * EP;   // row of a wavefront's block on its way to c in bytes, and all of them
  static constexpr int LDS = NST * STAGE > EPB ? NST * STAGE : EPB;
};

struct GGUnit { int g, rb, re, tm, tn, s0, s1, piece; bool on; };   // slices s0..s1 of tile (tm, tn) of group g

// Unit `id` (a tile, or one k piece of it) of the product.
template <int FORM, int BM, int BN>
__device__ __forceinline__ GGUnit gg_t_unit(const GGParams &p, int id) {
  GGUnit u{};
  const int base = gg_off(p, 0);
  int t, tiles_m, ntiles, nsl = 0, pieces;
  GGGroupTable gt{};
  if constexpr (FORM == 2) {
    tiles_m = p.tiles_m;
    ntiles = tiles_m * p.tiles_n * p.groups;
    pieces = p.pieces;
  } else {
    gt = gg_group_table<BM>(p, base, tiles_m);
    ntiles = tiles_m * p.tiles_n;
    nsl = (int)((p.k_dim + 63) / 64);
    pieces = p.sk_grid > 0 ? gg_t_pieces(p.sk_grid, ntiles, nsl) : 1;
  }
  u.on = id < ntiles * pieces;
  if (!u.on) return u;
  const int w = gg_xcd_chunk(id, ntiles * pieces);
  u.piece = __builtin_amdgcn_readfirstlane(w / ntiles);
  t = w - u.piece * ntiles;
  if constexpr (FORM == 2) {
    u.g = __builtin_amdgcn_readfirstlane(t / (tiles_m * p.tiles_n));
    t -= u.g * tiles_m * p.tiles_n;
    gg_tile_of(t, tiles_m, p.tiles_n, u.tm, u.tn);
    u.rb = gg_clamp_row(gg_off(p, u.g) - base, p.max_rows);
    u.re = gg_clamp_row(gg_off(p, u.g + 1) - base, p.max_rows);
    nsl = u.re > u.rb ? (u.re - u.rb + 63) / 64 : 0;
  } else {
    int tm_all;
    gg_tile_of(t, tiles_m, p.tiles_n, tm_all, u.tn);
    tm_all = __builtin_amdgcn_readfirstlane(tm_all);
    gg_locate<BM>(gt, tm_all, u.g, u.rb, u.re, u.tm);
  }
  u.tm = __builtin_amdgcn_readfirstlane(u.tm);
  u.tn = __builtin_amdgcn_readfirstlane(u.tn);
  u.s0 = __builtin_amdgcn_readfirstlane((int)((int64_t)u.piece * nsl / pieces));
  u.s1 = __builtin_amdgcn_readfirstlane((int)((int64_t)(u.piece + 1) * nsl / pieces));
  u.piece = pieces == 1 ? -1 : w;                                 // its place in the workspace
  return u;
}

template <typename T, int FORM, int BM, int BN, int ST>
__global__ void __launch_bounds__(2 * BN, ST == 1 ? 4 : 2) grouped_gemm_t_kernel(const GGParams p) {
  using C = GGT<FORM, BM, BN, ST>;
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr bool AKS = C::AKS, BKS = C::BKS;
  constexpr int MI = C::MI, NI = C::NI;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int wm = w / C::WN, wn = w % C::WN;

  // rows of c past the last group, up to max_rows, are zeroed here
  if constexpr (!AKS) {
    const int first = gg_clamp_row(gg_off(p, p.groups) - gg_off(p, 0), p.max_rows);
    const int nv = (int)(p.n_dim / 8);
    for (int r = first + (int)blockIdx.x; r < p.max_rows; r += (int)gridDim.x) {
      T *row = reinterpret_cast<T *>(p.c) + (int64_t)r * p.ldc;
      for (int v = tid; v < nv; v += 2 * BN) *reinterpret_cast<dh_u32x4 *>(row + 8 * v) = dh_u32x4{0u, 0u, 0u, 0u};
    }
  }
  const GGUnit u = gg_t_unit<FORM, BM, BN>(p, (int)blockIdx.x);
  if (!u.on) return;

  const int n0 = u.tn * BN, m0 = AKS ? u.tm * BM : u.rb + u.tm * BM;
  const int a_rext = AKS ? (int)(p.m_dim - m0) : u.re - m0, b_rext = (int)(p.n_dim - n0);
  const uint32_t lda_b = (uint32_t)p.lda * (uint32_t)sizeof(T), ldb_b = (uint32_t)p.ldb * (uint32_t)sizeof(T);
  const char *ag = reinterpret_cast<const char *>(p.a) + (AKS ? (int64_t)u.rb * lda_b + (int64_t)m0 * 2 : (int64_t)m0 * lda_b);
  const char *bg = reinterpret_cast<const char *>(p.b) +
                   (AKS ? (int64_t)u.rb * ldb_b + (int64_t)n0 * 2
                        : (int64_t)u.g * p.b_group_stride * 2 + (BKS ? (int64_t)n0 * 2 : (int64_t)n0 * ldb_b));
  const int64_t k_total = AKS ? u.re - u.rb : p.k_dim;
  const int64_t a_len = AKS ? k_total * lda_b - (int64_t)m0 * 2 : (int64_t)(a_rext < BM ? a_rext : BM) * lda_b;
  const int64_t b_len = BKS ? k_total * ldb_b - (int64_t)n0 * 2 : (int64_t)(b_rext < BN ? b_rext : BN) * ldb_b;
  const int64_t kstep_a = AKS ? (int64_t)64 * lda_b : 128, kstep_b = BKS ? (int64_t)64 * ldb_b : 128;

  // ---- copies: block b of a k-contiguous tile is 8 rows (a lane: row lane / 8, chunk lane % 8), of a k-strided one
  // 4 k rows (row lane / 16, chunk lane % 16); a wavefront takes neighbouring blocks
  constexpr uint32_t OUT = 0x80000000u;                           // a lane offset that is past any descriptor's end
  uint32_t va[C::ACPW], vb[C::BCPW];                              // lane offsets of this wavefront's copies
  {
    const int r8 = lane >> 3, ch = (lane & 7) ^ (r8 >> 1), r4 = lane >> 4, cs = (lane & 15) ^ (4 * r4);
#pragma unroll
    for (int x = 0; x < C::ACPW; ++x) {
      const int b = w * C::ACPW + x;
      va[x] = AKS ? (uint32_t)r4 * lda_b + (uint32_t)((cs ^ (b & 3)) << 4) : (uint32_t)r8 * lda_b + (uint32_t)((ch ^ (4 * (b & 1))) << 4);
    }
#pragma unroll
    for (int x = 0; x < C::BCPW; ++x) {
      const int b = w * C::BCPW + x;
      vb[x] = BKS ? (uint32_t)r4 * ldb_b + (uint32_t)((cs ^ (b & 3)) << 4) : (uint32_t)r8 * ldb_b + (uint32_t)((ch ^ (4 * (b & 1))) << 4);
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int kc_tail = (int)(k_total % 64);                        // k-contiguous operands: chunks past it read as zero
  int4v ra, rb;
  auto descriptors = [&](int s) {
    ra = raw_rsrc(ag + s * kstep_a, a_len - s * kstep_a);
    rb = raw_rsrc(bg + s * kstep_b, b_len - s * kstep_b);
    asm volatile("s_nop 4" : "+s"(ra), "+s"(rb));                 // readfirstlane -> memory instruction
  };
  // copy x (of C::CPW) of slice s into stage st
  auto copy = [&](int x, int s, uint32_t stage) {
    const bool tail = !(AKS && BKS) && kc_tail != 0 && (s + 1) * 64 > (int)k_total;
    if (x < C::ACPW) {
      const int b = w * C::ACPW + x;                              // block of the A tile
      uint32_t v = va[x];
      if (!AKS && tail) {
        const int ch = ((lane & 7) ^ (lane >> 4)) ^ (4 * (b & 1));
        if (ch * 8 >= kc_tail) v = OUT;
      }
      copy_1k(v, ra, (uint32_t)((AKS ? 4 : 8) * b) * lda_b, stage + (uint32_t)(b * 1024));
    } else {
      const int y = x - C::ACPW, b = w * C::BCPW + y;             // (a k-strided B tile of 256 columns is two of 128)
      uint32_t v = vb[y];
      if (!BKS && tail) {
        const int ch = ((lane & 7) ^ (lane >> 4)) ^ (4 * (b & 1));
        if (ch * 8 >= kc_tail) v = OUT;
      }
      const uint32_t off = BKS ? (uint32_t)(4 * (b & 15)) * ldb_b + (uint32_t)((b >> 4) * 256) : (uint32_t)(8 * b) * ldb_b;
      copy_1k(v, rb, off, stage + (uint32_t)(C::ABYTES + b * 1024));
    }
  };

  // ---- fragments
  const uint32_t sw = (uint32_t)((hh ^ ((c >> 1) & 7)) << 4);
  const uint32_t fa_lane = (uint32_t)((wm * 32 * MI + c) * 128) + sw, fb_lane = (uint32_t)(C::ABYTES + (wn * 32 * NI + c) * 128) + sw;
  const int r16 = lane & 15, t_lc = 2 * ((lane >> 4) & 1) + ((r16 & 3) >> 1), tx = 4 * (r16 >> 2) + 2 * hh;
  const uint32_t t_row = (uint32_t)((8 * hh + (r16 >> 2)) * 256 + (r16 & 1) * 8);
  const uint32_t t_lo = t_row + (uint32_t)((t_lc ^ tx) << 4), t_hi = t_row + 1024 + (uint32_t)((t_lc ^ (tx + 1)) << 4);
  typedef __attribute__((address_space(3))) const Frag *lds_frag;
  typedef short4v __attribute__((address_space(3))) *lds_tr;
  auto tr_frag = [&](uint32_t tile, int blk, int ks) {            // 32 columns `blk` of a k-strided tile, k step ks
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(tile + (t_lo ^ (uint32_t)(blk << 6)) + (uint32_t)(ks * 4096)));
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(tile + (t_hi ^ (uint32_t)(blk << 6)) + (uint32_t)(ks * 4096)));
    return frag_join<T>(lo, hi);
  };
  auto frag_a = [&](uint32_t stage, int i, int ks) -> Frag {
    if constexpr (AKS) return tr_frag(stage, wm * MI + i, ks);
    else return *(lds_frag)(stage + (fa_lane ^ (uint32_t)(ks << 5)) + (uint32_t)(i * 4096));
  };
  auto frag_b = [&](uint32_t stage, int j, int ks) -> Frag {
    if constexpr (BKS) return tr_frag(stage + C::ABYTES + (uint32_t)((wn * NI + j) / 4 * 16384), (wn * NI + j) % 4, ks);
    else return *(lds_frag)(stage + (fb_lane ^ (uint32_t)(ks << 5)) + (uint32_t)(j * 4096));
  };

  floatx16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // Slice s lies in stage s % NST.  At its head a wavefront waits for its own copies of it (those of the NST - 2 slices
  // behind it stay in flight) and for its LDS reads of the slice before, and meets the others; then slice s + NST - 1 may
  // overwrite the stage of slice s - 1.  Fragments are read one k step (16) ahead.
  const int cnt = u.s1 - u.s0;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (the zeroed rows' stores are not part of the counts below)
#pragma unroll
  for (int i = 0; i < C::NST - 1; ++i)
    if (i < cnt) {
      descriptors(u.s0 + i);
#pragma unroll
      for (int x = 0; x < C::CPW; ++x) copy(x, u.s0 + i, lds0 + (uint32_t)(i * C::STAGE));
    }
  int st = 0;
  auto slice = [&](auto morec, int s) {
    constexpr bool MORE = decltype(morec)::value;                 // slice s + NST - 1 exists
    if (C::NST > 1 && (MORE || s + C::NST - 2 < cnt)) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::NST > 1 ? (C::NST - 2) * C::CPW : 0) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint32_t cur = lds0 + (uint32_t)(st * C::STAGE);
    const uint32_t free = lds0 + (uint32_t)((st == 0 ? C::NST - 1 : st - 1) * C::STAGE);   // stage of slices s - 1 and s + NST - 1
    st = st + 1 == C::NST ? 0 : st + 1;
    const int sn = u.s0 + s + C::NST - 1;
    if (MORE) descriptors(sn);
    Frag fa[2][MI], fb[2][NI];
    auto frags = [&](int ks) {
#pragma unroll
      for (int j = 0; j < NI; ++j) fb[ks & 1][j] = frag_b(cur, j, ks);
#pragma unroll
      for (int i = 0; i < MI; ++i) fa[ks & 1][i] = frag_a(cur, i, ks);
    };
    frags(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) frags(ks + 1);
      if (MORE) {
#pragma unroll
        for (int x = ks * C::CPW / 4; x < (ks + 1) * C::CPW / 4; ++x) copy(x, sn, free);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = M::mma(fb[ks & 1][j], fa[ks & 1][i], acc[i][j]);   // C^T: lane column = output row
    }
  };
  int s = 0;
  if constexpr (C::NST == 1) {                                    // what is in flight is the other workgroups' business
#pragma unroll 1
    for (; s < cnt; ++s) {
      if (s > 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      descriptors(u.s0 + s);
#pragma unroll
      for (int x = 0; x < C::CPW; ++x) copy(x, u.s0 + s, lds0);
      slice(std::false_type{}, s);
    }
  } else {
#pragma unroll 1
    for (; s + C::NST - 1 < cnt; ++s) slice(std::true_type{}, s);
#pragma unroll 1
    for (; s < cnt; ++s) slice(std::false_type{}, s);
  }

  if (u.piece >= 0) {                                             // fp32 piece in accumulator layout, 1 KB per instruction
    float *dst = p.ws + (size_t)u.piece * (BM * BN) + (size_t)(w * MI * NI) * 1024 + (size_t)lane * 4;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 o = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<floatx4 *>(dst + (i * NI + j) * 1024 + q * 256) = o;
        }
    return;
  }
  T *cg = reinterpret_cast<T *>(p.c) + (AKS ? (int64_t)u.g * p.c_group_stride : 0) + (int64_t)m0 * p.ldc + n0;
  struct alignas(8) Q4 { T v[4]; };
  if (AKS && p.accumulate) {                                      // c += product, one rounding
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = wm * 32 * MI + 32 * i + c;
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = wn * 32 * NI + 32 * j + 8 * q + 4 * hh;
          if (m < a_rext && n < b_rext) {
            Q4 *dst = reinterpret_cast<Q4 *>(cg + (int64_t)m * p.ldc + n);
            const Q4 old = *dst;
            Q4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[i][j][4 * q + e] + static_cast<float>(old.v[e]));
            *dst = o;
          }
        }
    }
    return;
  }
  // whole row segments of the wavefront's block through its own LDS region (rows 8 bytes apart in the banks)
  constexpr int EP = C::EP, LPR = NI * 4;                         // region row in bytes, lanes per row of 16-byte pieces
  __syncthreads();                                                // everyone is done with the stages
  unsigned char *ep = smem + w * (32 * MI * EP);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        Q4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[i][j][4 * q + e]);
        *reinterpret_cast<Q4 *>(ep + (32 * i + c) * EP + (32 * j + 8 * q + 4 * hh) * 2) = o;
      }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  const int er = lane / LPR, ec = lane % LPR;
#pragma unroll
  for (int it = 0; it < 32 * MI * LPR / 64; ++it) {
    const int r = it * (64 / LPR) + er, m = wm * 32 * MI + r, n = wn * 32 * NI + 8 * ec;
    const dh_u32x4 o = *reinterpret_cast<const dh_u32x4 *>(ep + r * EP + ec * 16);
    if (m < a_rext && n < b_rext) *reinterpret_cast<dh_u32x4 *>(cg + (int64_t)m * p.ldc + n) = o;
  }
}

// Sums the k pieces of grouped_gemm_t_kernel's tiles in k order and stores the tiles: a wavefront per 32x32 block.
template <typename T, int FORM, int BM, int BN>
__global__ void __launch_bounds__(256) gg_t_reduce_kernel(const GGParams p) {
  using C = GGT<FORM, BM, BN>;
  constexpr int BLOCKS = BM * BN / 1024;                          // 32x32 blocks of a tile
  const int lane = threadIdx.x & 63, base = gg_off(p, 0);
  const int id = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = id / BLOCKS, blk = id % BLOCKS;
  int ntiles, tm, tn, rb, re, g, pieces;
  if constexpr (FORM == 2) {
    ntiles = p.tiles_m * p.tiles_n * p.groups;
    pieces = p.pieces;
    if (t >= ntiles) return;
    g = t / (p.tiles_m * p.tiles_n);
    gg_tile_of(t - g * p.tiles_m * p.tiles_n, p.tiles_m, p.tiles_n, tm, tn);
    rb = 0;
    re = (int)p.m_dim;
  } else {
    int tiles_m, tm_all;
    const GGGroupTable gt = gg_group_table<BM>(p, base, tiles_m);
    ntiles = tiles_m * p.tiles_n;
    pieces = gg_t_pieces(p.sk_grid, ntiles, (int)((p.k_dim + 63) / 64));
    if (t >= ntiles || pieces == 1) return;
    gg_tile_of(t, tiles_m, p.tiles_n, tm_all, tn);
    tm_all = __builtin_amdgcn_readfirstlane(tm_all);
    gg_locate<BM>(gt, tm_all, g, rb, re, tm);
    g = 0;
  }
  floatx4 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int pc = 0; pc < pieces; ++pc) {
    const float *src = p.ws + (size_t)(pc * ntiles + t) * (BM * BN) + (size_t)blk * 1024 + (size_t)lane * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] += *reinterpret_cast<const floatx4 *>(src + q * 256);
  }
  const int w = blk / (C::MI * C::NI), i = blk / C::NI % C::MI, j = blk % C::NI;
  const int m = rb + tm * BM + (w / C::WN * C::MI + i) * 32 + (lane & 31), n = tn * BN + (w % C::WN * C::NI + j) * 32 + 4 * (lane >> 5);
  if (m >= re) return;
  T *dst = reinterpret_cast<T *>(p.c) + (FORM == 2 ? (int64_t)g * p.c_group_stride : 0) + (int64_t)m * p.ldc + n;
  struct alignas(8) Q4 { T v[4]; };
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (n + 8 * q < p.n_dim) {
      Q4 o;
      if (FORM == 2 && p.accumulate) {
        const Q4 old = *reinterpret_cast<const Q4 *>(dst + 8 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[q][e] + static_cast<float>(old.v[e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[q][e]);
      }
      *reinterpret_cast<Q4 *>(dst + 8 * q) = o;
    }
}

// Rows longer than GG_MAX_LD elements, whose tiles do not fit the 31-bit byte offsets of the kernels above: a wavefront per
// row and 8 columns of c, its lanes share the reduction, 64-bit addresses.  Bound by the rate of its loads; such operands
// are only ever a few rows.
template <typename T, int FORM>
__global__ void __launch_bounds__(256) grouped_gemm_long_rows_kernel(const GGParams p) {
  using V = Vec<T>;
  const int lane = threadIdx.x & 63, base = gg_off(p, 0);
  const T *a = reinterpret_cast<const T *>(p.a), *b = reinterpret_cast<const T *>(p.b);
  T *c = reinterpret_cast<T *>(p.c);
  const int64_t cols = p.n_dim / 8, rows = FORM == 2 ? p.m_dim * p.groups : p.max_rows;
  for (int64_t it = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); it < rows * cols; it += (int64_t)gridDim.x * 4) {
    const int64_t row = it / cols, n = 8 * (it - row * cols);
    int64_t k0 = 0, k1 = 0;                                       // the reduction: columns of a, or rows (TN)
    const T *ar = a, *bg = b;
    int64_t astep = 1;
    T *dst;
    if constexpr (FORM == 2) {
      const int g = (int)(row / p.m_dim);
      const int64_t m = row - (int64_t)g * p.m_dim;
      k0 = gg_clamp_row(gg_off(p, g) - base, p.max_rows);
      k1 = gg_clamp_row(gg_off(p, g + 1) - base, p.max_rows);
      ar = a + m;
      astep = p.lda;
      dst = c + (int64_t)g * p.c_group_stride + m * p.ldc + n;
    } else {
      ar = a + row * p.lda;
      dst = c + row * p.ldc + n;
      for (int g = 0; g < p.groups; ++g)                          // rows past the last group: zeros
        if (row >= gg_clamp_row(gg_off(p, g) - base, p.max_rows) && row < gg_clamp_row(gg_off(p, g + 1) - base, p.max_rows)) {
          bg = b + (int64_t)g * p.b_group_stride;
          k1 = p.k_dim;
        }
    }
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int64_t k = k0 + lane; k < k1; k += 64) {
      const float x = to_f(ar[k * astep]);
      if constexpr (FORM == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += x * to_f(bg[(n + j) * p.ldb + k]);
      } else {
        const V v = ldg(bg + k * p.ldb + n);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += x * to_f(v.v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      for (int o = 32; o > 0; o >>= 1) acc[j] += __shfl_xor(acc[j], o, 64);
    if (lane == 0) {
      V o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o.v[j] = static_cast<T>(FORM == 2 && p.accumulate ? acc[j] + to_f(dst[j]) : acc[j]);
      stg(dst, o);
    }
  }
}

// Workspace of the split last round: one fp32 tile per workgroup of the grid.
constexpr int GG_SK_MAX_GRID = 256;
constexpr size_t GG_SK_WS_BYTES = (size_t)GG_SK_MAX_GRID * 256 * 256 * sizeof(float);

// Compute units of the current device (asked for once per device).
static int gg_compute_units(int &cus) {
  static std::atomic<int> known[64];
  int dev = 0;
  DH_HIP(hipGetDevice(&dev));
  cus = known[dev & 63].load(std::memory_order_relaxed);
  if (cus == 0) {
    DH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    known[dev & 63].store(cus, std::memory_order_relaxed);
  }
  return DH_OK;
}

template <typename T>
static int launch_gg_w8_tn(GGParams p, hipStream_t st) {
  p.tiles_m = (int)cdiv(p.m_dim, 256);
  p.tiles_n = (int)cdiv(p.n_dim, 256);
  hipLaunchKernelGGL((grouped_gemm_w8_kernel<T, 2, false>), dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.groups), dim3(512), 0, st, p);
  return DH_OK;
}

template <typename T, bool BKS>
static int launch_gg_w8(GGParams p, int64_t m_extent, void *workspace, size_t workspace_bytes, hipStream_t st) {
  p.tiles_n = (int)cdiv(p.n_dim, 256);
  p.tiles_m = (int)(cdiv(m_extent, 256) + p.groups);
  if (p.tiles_m <= 0 || p.tiles_n <= 0) return DH_OK;
  p.zero_tail = 1;
  int grid = 0;
  if (workspace != nullptr && p.k_dim >= 64) {
    int cus = 0;
    const int rc = gg_compute_units(cus);
    if (rc) return rc;
    grid = cus < GG_SK_MAX_GRID ? cus : GG_SK_MAX_GRID;
    if (workspace_bytes < (size_t)grid * 256 * 256 * sizeof(float)) grid = 0;
  }
  // With a workspace the last round of tiles may be split along k (decided on the device, where the tile count is
  // known) by up to `grid` workgroups more.  Where nothing is split the sum's launch is for nothing (5 us); a split saves up to
  // half a tile time (45 us and more).
  p.sk_grid = grid;
  if (grid == 0) {
    hipLaunchKernelGGL((grouped_gemm_w8_kernel<T, BKS ? 1 : 0, false>), dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(512), 0, st, p);
    return DH_OK;
  }
  p.ws = reinterpret_cast<float *>(workspace);
  hipLaunchKernelGGL((grouped_gemm_w8_kernel<T, BKS ? 1 : 0, true>), dim3((unsigned)(p.tiles_m * p.tiles_n + grid)), dim3(512), 0, st, p);
  hipLaunchKernelGGL((gg_split_reduce_kernel<T>), dim3((unsigned)(16 * grid / 2)), dim3(256), 0, st, p, grid);   // at most grid / 2 tiles are split
  return DH_OK;
}

template <typename T, int FORM, int BM, int BN, int ST = 0>
static int launch_gg_t(GGParams p, int64_t m_extent, void *workspace, size_t workspace_bytes, hipStream_t st) {
  using C = GGT<FORM, BM, BN, ST>;
  constexpr int BLOCKS = BM * BN / 1024;
  int cus = 0;
  const int rc = gg_compute_units(cus);
  if (rc) return rc;
  int slots = C::PER_CU * (cus < GG_SK_MAX_GRID ? cus : GG_SK_MAX_GRID);
  if (workspace == nullptr || workspace_bytes < (size_t)slots * BM * BN * sizeof(float)) slots = 0;
  p.ws = reinterpret_cast<float *>(workspace);
  p.tiles_n = (int)cdiv(p.n_dim, BN);
  p.tiles_m = (int)cdiv(m_extent, BM);
  p.sk_grid = 0;
  p.pieces = 1;
  int64_t grid, reduce = 0;
  if (FORM == 2) {
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n * p.groups;
    if (slots > 0) p.pieces = gg_t_pieces(slots, (int)(tiles < slots ? tiles : slots), (int)cdiv(cdiv(p.max_rows, p.groups), 64));
    grid = tiles * p.pieces;
    if (p.pieces > 1) reduce = tiles;
  } else {
    const int64_t most = ((int64_t)p.tiles_m + p.groups) * p.tiles_n;       // every group may end in a part of a tile
    grid = most;
    // the pieces are chosen on the device, where the tile count is known; not at all where it cannot be small
    if ((int64_t)p.tiles_m * p.tiles_n * 2 <= slots && p.k_dim >= 16 * 64) {
      p.sk_grid = slots;
      if (grid < slots) grid = slots;
      reduce = most < slots / 2 ? most : slots / 2;
    }
  }
  DH_CHECK(grid > 0 && grid < (1ll << 31), "grouped GEMM: too many tiles");
  hipLaunchKernelGGL((grouped_gemm_t_kernel<T, FORM, BM, BN, ST>), dim3((unsigned)grid), dim3(2 * BN), 0, st, p);
  if (reduce > 0)
    hipLaunchKernelGGL((gg_t_reduce_kernel<T, FORM, BM, BN>), dim3((unsigned)cdiv(reduce * BLOCKS, 4)), dim3(256), 0, st, p);
  return DH_OK;
}

// Row tiles of `bm` that rows in `groups` uneven groups come to: the mean of groups of the average size and of one standard
// deviation of a random routing above and below it.
static double gg_tiles(int64_t rows, int groups, int bm) {
  const double avg = (double)rows / groups, dev = groups > 1 ? std::sqrt(avg) : 0;
  return groups * (std::ceil((avg - dev) / bm) + std::ceil(avg / bm) + std::ceil((avg + dev) / bm)) / 3;
}

template <typename T, int FORM>
static int dispatch_gg_t(const GGParams &p, int64_t m_extent, void *workspace, size_t workspace_bytes, hipStream_t st) {
  // (the columns of an NT product are no row length of an operand: only their tiles are counted in 32 bits)
  if (p.n_dim > (FORM == 0 ? (int64_t)1 << 30 : GG_MAX_LD) || (FORM == 2 ? p.m_dim : p.k_dim) > GG_MAX_LD) {
    const int64_t items = (FORM == 2 ? p.m_dim * p.groups : (int64_t)p.max_rows) * (p.n_dim / 8);
    const int64_t blocks = cdiv(items, 4) < 256 * 16 ? cdiv(items, 4) : 256 * 16;
    hipLaunchKernelGGL((grouped_gemm_long_rows_kernel<T, FORM>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    return DH_OK;
  }
  if constexpr (FORM == 2) {
    // (the one-stage form: above.  Accumulating, only products of few tiles and narrow ones come here)
    if (!p.accumulate && p.groups * cdiv(p.m_dim, 128) * cdiv(p.n_dim, 128) > 512)
      return launch_gg_t<T, FORM, 128, 128, 1>(p, m_extent, workspace, workspace_bytes, st);
    return launch_gg_t<T, FORM, 128, 128>(p, m_extent, workspace, workspace_bytes, st);
  } else {
    // Rows per tile.  Small ones where a group's rows fit one tile (weights are then read once, by more workgroups the
    // narrower the tile), and where tiles of 128 rows are so few that 64-row ones fill the 512 places better: fewer than half
    // of them (then they are split along k), or about all of them, or, for reductions that the larger tiles cannot split
    // either, anything in between.  us for 32 / 64 / 128 rows, n = 2048 of 1408, 8 groups: 24 rows a group 12.3 / 14.2 / 23.6,
    // 48 rows 12.6 / 14.3 / 23.9, 128 rows 21.6 / 19.3 / 24.7; 64 groups, n = 1024 of 704: 16 rows 15.8 / 16.0 / 16.2, 48 rows
    // 20.3 / 17.0 / 17.2, 100 rows 31.7 / 23.4 / 20.0.  64-row tiles / the better of 128x128 and 128x256, by their number and k:
    // 256, 1408 15.8 / 24.5; 288, 2048 24.4 / 27.7; 384, 2816 33.3 / 38.9; 448, 1408 17.8 / 25.5; but 256, 2816 (2000 rows) 4 us
    // more; 256, 7168 71.6 / 47.5; 512, 5632 91.1 / 74.9; 528, 2048 43.6 / 31.8.  Over 360 products of 16 to 65536 rows the tile
    // picked here is 3.5 % from the best of the five kernels on average.
    const int64_t avg = m_extent / p.groups;
    const int64_t tiles64 = p.groups * (avg / 64 + 1) * cdiv(p.n_dim, 128);
    const bool few = p.groups * cdiv(avg, 128) * cdiv(p.n_dim, 128) < 400;
    if (avg <= 24 || (few && avg <= 56)) return launch_gg_t<T, FORM, 32, 128>(p, m_extent, workspace, workspace_bytes, st);
    if (avg <= 56 || (few && (tiles64 <= 224 || (tiles64 <= 512 && p.k_dim <= (tiles64 > 340 ? 3072 : 2048)))))
      return launch_gg_t<T, FORM, 64, 128>(p, m_extent, workspace, workspace_bytes, st);
    // long reductions: 128x256 tiles move a quarter less through L2 per product (3062 rows of 8 groups, n = 4096 of 5632:
    // 202 -> 178 us); short ones cannot hide the first loads and last stores of their single workgroup per compute unit
    // (16384 rows, n = 1408 of 1024: 60 -> 71 us)
    if (p.k_dim >= 1536) return launch_gg_t<T, FORM, 128, 256>(p, m_extent, workspace, workspace_bytes, st);
    // more tiles than two workgroups on every compute unit take: the one-stage form, us two stages / one, 8 groups, n = 5632 of
    // 1024: 128 rows a group (528 tiles) 36 / 31, 1024 125 / 105; 64 groups, n = 1408 of 1024: 72 rows (748) 39 / 37, 256 79 / 67; 16
    // groups, n = 1408 of 512: 256 rows (440) 14.5 / 16.3, 384 (616) 22.4 / 19.8.  Of longer reductions 128x256 tiles run better
    if (gg_tiles(m_extent, p.groups, 128) * (double)cdiv(p.n_dim, 128) > 512)
      return launch_gg_t<T, FORM, 128, 128, 1>(p, m_extent, workspace, workspace_bytes, st);
    return launch_gg_t<T, FORM, 128, 128>(p, m_extent, workspace, workspace_bytes, st);
  }
}

// NT / NN: whether 256x256 tiles, one workgroup per compute unit, are the faster ones.  All kernels run in rounds of equal
// tiles, so the times follow from the number of rounds (the last one of the 256x256 tiles is split along k where it is at
// most half full; the one-stage form's rounds run into each other) and of k slices; the constants (us) are least-squares fits
// to 330 products of 1 to 64 groups, 192 to 4096 rows a group, n and k from 512 to 8192, which the formulas meet to 13 and 11 %.
// Rows that are routed at random fill more tiles than groups of their average (gg_tiles).  256x256 / smaller, us: 16 groups of 128
// rows, n = 4096 of 2816 93 / 104, of 72 rows 86 / 76, of 384 154 / 164 (groups of 360 to 410 rows: 2 tiles of 256, 3 or 4 of 128); 2 x
// 640, n = 7168 of 4096 80 / 112, 2 x 256 52 / 44; 8 x 1024, n = 5632 of 1024 126 / 105, n = 1024 of 2816 62 / 80.  Many groups of few rows
// read their weights too slowly in large tiles for the formula: 64 groups, n = 1024 of 2048: 128 rows 102 / 81, 256 167 / 112, 384 150
// / 152, 640 181 / 243.
static bool gg_w8_pays(int64_t rows, int groups, int64_t n, int64_t k) {
  const int64_t avg = rows / groups;
  if (avg < 96 || avg < 6 * groups) return false;
  const double ns = (double)cdiv(k, 64);
  const int64_t tiles = (int64_t)std::ceil(gg_tiles(rows, groups, 256)) * cdiv(n, 256), rem = tiles % 256;
  const double round = 14.3 + 1.357 * ns;
  double big = 4.6 + (double)(tiles / 256) * round;
  if (rem > 128) big += round;
  else if (rem > 0) big += 26.3 + 1.357 * (ns > 1 ? ns / (double)(256 / rem < ns ? 256 / rem : ns) : 1.0);
  double small;
  if (k >= 1536) {
    const int64_t t = (int64_t)std::ceil(gg_tiles(rows, groups, 128)) * cdiv(n, 256);
    if (2 * t <= 256) small = 15.4 + 0.932 * ns * (double)t / 256;
    else if (t < 256) small = 9.4 + 0.932 * ns * (0.25 + 0.75 * (double)t / 256);
    else small = (double)cdiv(t, 256) * (9.4 + 0.932 * ns);
  } else {
    const double t = gg_tiles(rows, groups, 128) * (double)cdiv(n, 128), part = t / 512 > 8 / ns ? t / 512 : 8 / ns;
    small = 2 * t <= 512 ? 6 + 1.205 * ns * part : t <= 512 ? 1.205 * ns : 6 + 2.3 * ns * t / 1024;
  }
  return big < small;
}

// The same for TN (constants from 80 products of 16 to 2048 rows a group; below six slices, where uneven groups add some, 10 % is
// asked for); us, 256x256 / 128x128 tiles: 16 groups of 5632 x 4096: 192 rows 275 / 289, 512 452 / 496, 1024 726 / 844; 8 groups of 5632 x
// 1024: 256 rows 47 / 41, 1024 100 / 104.  Accumulating, which the smaller tiles do with 8-byte accesses, from two thirds of a
// tile for every compute unit on: 16 groups of 5632 x 4096: 16 rows 267 / 569, 256 364 / 684; of 1408 x 512 (192 tiles) 11 / 20, 18 / 27; one
// group of 16 rows, 4096 x 4096 13 / 33, of 256 rows, 1280 x 8192 15 / 24, but 8192 x 1024 (128 tiles) 15 / 16, of 4096 rows 84 / 74.  Not where
// most of a tile is past the matrix: as fast as the smaller ones where a third of it is output (500 products of up to 480 columns
// the narrow way; up to a tenth 0.58 of their speed, to 0.2 0.8, to 0.3 0.9, 0.3 to 0.4 1.0, 0.5 to 0.6 1.17, beyond 0.7 1.5).
static bool gg_w8_tn_pays(int64_t rows, int groups, int64_t m, int64_t n, int accumulate) {
  const int64_t avg = rows / groups;
  const double ns = (double)cdiv(avg, 64);
  const int64_t tiles = groups * cdiv(m, 256) * cdiv(n, 256), small = groups * cdiv(m, 128) * cdiv(n, 128);
  if (accumulate && tiles >= 160 && 100 * m * n >= 35 * 65536 * (tiles / groups)) return true;
  if (avg < 192) return false;
  return (double)cdiv(tiles, 256) * (8.5 + 1.38 * ns) * (avg < 384 ? 1.1 : 1.0) <
         (accumulate || small <= 512 ? 0.8 + (double)small / 512 * (3.5 + 1.11 * ns) : (double)small / 1024 * (6.3 + 1.85 * ns));
}

// Tiles of a TN product: 256, 128 (dispatch_gg_t), or 0 (rows too long for tiles).  The offsets of the 256x256 tiles have to fit
// the 32-bit buffer addressing: of the operands, of the 64 rows of a slice, however few of them there are, and, accumulating, of
// a tile's 256 rows of c.  (Otherwise the rows that gg_w8_tn_pays asks for keep them short.)
static int gg_tn_tiles(int64_t rows, int groups, int64_t m, int64_t n, int accumulate) {
  const bool fits = rows * (m > n ? m : n) * 2 < (1ll << 31) && (!accumulate || (m <= GG_MAX_LD && n <= GG_MAX_LD));
  if (fits && gg_w8_tn_pays(rows, groups, m, n, accumulate)) return 256;
  return m > GG_MAX_LD || n > GG_MAX_LD ? 0 : 128;
}

static int gg_common_checks(const void *a, const void *b, void *c, const int32_t *offs, int groups, int dtype) {
  DH_CHECK(groups >= 1 && groups <= GG_MAX_GROUPS, "groups=%d must be in [1, %d]", groups, GG_MAX_GROUPS);
  DH_CHECK(dtype == DH_BF16 || dtype == DH_F16, "grouped GEMM supports bf16/fp16 (dtype %d)", dtype);
  DH_CHECK(a && b && c && (offs || groups == 1), "null pointer");
  DH_CHECK(aligned16(a) && aligned16(b) && aligned16(c), "operands must be 16-byte aligned");
  return DH_OK;
}

}  // namespace dh

extern "C" size_t dh_grouped_gemm_workspace_bytes(void) { return dh::GG_SK_WS_BYTES; }

extern "C" int dh_grouped_gemm_nt(const void *a, const void *b, void *c, const int32_t *offs, int groups,
                                  int64_t max_rows, int64_t n, int64_t k, int dtype, void *workspace,
                                  size_t workspace_bytes, void *stream) {
  using namespace dh;
  DH_CHECK(max_rows >= 0 && max_rows < (1ll << 31) && n >= 0 && k >= 0, "size out of range");
  if (max_rows == 0 || n == 0) return DH_OK;
  int rc = gg_common_checks(a, b, c, offs, groups, dtype);
  if (rc) return rc;
  DH_CHECK(n % 8 == 0 && k % 8 == 0, "n=%lld and k=%lld must be multiples of 8", (long long)n, (long long)k);
  GGParams p{};
  p.a = a; p.b = b; p.c = c; p.offs = offs; p.groups = groups;
  p.n_dim = n; p.k_dim = k; p.lda = k; p.ldb = k; p.ldc = n;
  p.b_group_stride = n * k; p.accumulate = 0; p.max_rows = (int)max_rows;
  const bool big = gg_w8_pays(max_rows, groups, n, k);
  if (big && k <= (1ll << 21)) {
    rc = dtype == DH_BF16 ? launch_gg_w8<bf16_t, false>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : launch_gg_w8<f16_t, false>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
  } else {
    rc = dtype == DH_BF16 ? dispatch_gg_t<bf16_t, 0>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : dispatch_gg_t<f16_t, 0>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
  }
  if (rc) return rc;
  DH_LAUNCH_CHECK();
  return DH_OK;
}

extern "C" int dh_grouped_gemm_nn(const void *a, const void *b, void *c, const int32_t *offs, int groups,
                                  int64_t max_rows, int64_t n, int64_t k, int dtype, void *workspace,
                                  size_t workspace_bytes, void *stream) {
  using namespace dh;
  DH_CHECK(max_rows >= 0 && max_rows < (1ll << 31) && n >= 0 && k >= 0, "size out of range");
  if (max_rows == 0 || n == 0) return DH_OK;
  int rc = gg_common_checks(a, b, c, offs, groups, dtype);
  if (rc) return rc;
  DH_CHECK(n % 8 == 0 && k % 8 == 0, "n=%lld and k=%lld must be multiples of 8", (long long)n, (long long)k);
  GGParams p{};
  p.a = a; p.b = b; p.c = c; p.offs = offs; p.groups = groups;
  p.n_dim = n; p.k_dim = k; p.lda = k; p.ldb = n; p.ldc = n;
  p.b_group_stride = n * k; p.accumulate = 0; p.max_rows = (int)max_rows;
  const bool big = gg_w8_pays(max_rows, groups, n, k);
  if (big && k <= (1ll << 21) && k * n * (int64_t)dtype_size(dtype) < (1ll << 31)) {
    rc = dtype == DH_BF16 ? launch_gg_w8<bf16_t, true>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : launch_gg_w8<f16_t, true>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
  } else {
    rc = dtype == DH_BF16 ? dispatch_gg_t<bf16_t, 1>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : dispatch_gg_t<f16_t, 1>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
  }
  if (rc) return rc;
  DH_LAUNCH_CHECK();
  return DH_OK;
}

extern "C" int dh_grouped_gemm_tn_ws(const void *a, const void *b, void *c, const int32_t *offs, int groups,
                                     int64_t max_rows, int64_t m, int64_t n, int accumulate, int dtype, void *workspace,
                                     size_t workspace_bytes, void *stream) {
  using namespace dh;
  DH_CHECK(max_rows >= 0 && max_rows < (1ll << 31) && n >= 0 && m >= 0, "size out of range");
  if (m == 0 || n == 0) return DH_OK;
  int rc = gg_common_checks(a, b, c, offs, groups, dtype);
  if (rc) return rc;
  DH_CHECK(n % 8 == 0 && m % 8 == 0, "m=%lld and n=%lld must be multiples of 8", (long long)m, (long long)n);
  GGParams p{};
  p.a = a; p.b = b; p.c = c; p.offs = offs; p.groups = groups;
  p.m_dim = m; p.n_dim = n; p.lda = m; p.ldb = n; p.ldc = n;
  p.c_group_stride = m * n; p.accumulate = accumulate; p.max_rows = (int)max_rows;
  if (gg_tn_tiles(max_rows, groups, m, n, accumulate) == 256)
    rc = dtype == DH_BF16 ? launch_gg_w8_tn<bf16_t>(p, (hipStream_t)stream) : launch_gg_w8_tn<f16_t>(p, (hipStream_t)stream);
  else
    rc = dtype == DH_BF16 ? dispatch_gg_t<bf16_t, 2>(p, m, workspace, workspace_bytes, (hipStream_t)stream)
                          : dispatch_gg_t<f16_t, 2>(p, m, workspace, workspace_bytes, (hipStream_t)stream);
  if (rc) return rc;
  DH_LAUNCH_CHECK();
  return DH_OK;
}

extern "C" int dh_grouped_gemm_tn_tiles(int groups, int64_t max_rows, int64_t m, int64_t n, int accumulate) {
  return groups < 1 || max_rows < 0 || m <= 0 || n <= 0 ? 0 : dh::gg_tn_tiles(max_rows, groups, m, n, accumulate);
}

extern "C" int dh_grouped_gemm_tn(const void *a, const void *b, void *c, const int32_t *offs, int groups,
                                  int64_t max_rows, int64_t m, int64_t n, int accumulate, int dtype, void *stream) {
  return dh_grouped_gemm_tn_ws(a, b, c, offs, groups, max_rows, m, n, accumulate, dtype, nullptr, 0, stream);
}
