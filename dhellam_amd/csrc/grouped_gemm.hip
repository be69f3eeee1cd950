// Grouped GEMM on gfx950 MFMA (bf16/fp16 inputs, fp32 accumulate) for one
// expert-parallel rank: every local expert multiplies its own contiguous block
// of permuted rows.
//
// One template covers the three products a SwiGLU expert needs:
//   NT  c[r, n]  = sum_k a[r, k] * w[g][n, k]      forward  (both k-contiguous)
//   NN  c[r, n]  = sum_k a[r, k] * w[g][k, n]      dgrad    (w strided in k)
//   TN  c[g][m,n] = sum_r a[r, m] * b[r, n]        wgrad    (both strided in k = r)
// Two kernels.  grouped_gemm_w4_kernel (products that fill the chip): 256x256 tiles, four wavefronts of 128x128 with
// hand-placed copies, optionally one workgroup per compute unit that takes whole tiles in rounds and a k piece of a tile
// of the last round.  grouped_gemm_t_kernel (everything else): smaller tiles, copied straight to LDS, split along k where
// there are few of them.  k-contiguous operands are read from LDS as 16-byte row fragments; k-strided operands stay
// row-major in LDS and are read with transpose loads, so no operand is ever transposed in memory.
// The product is formed as C^T (weights in the MFMA A slot) so that each lane
// ends up with runs of 4 consecutive output columns of one row: 8-byte stores.
// Group row ranges are read on the device from the offsets table.
#include "mma.h"
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
  int zero_tail;         // NT/NN on grouped_gemm_w4_kernel: the kernel itself zeroes the rows of c past the last group
  int sk_grid;           // grouped_gemm_w4_kernel: > 0: a split kernel of that many workgroups follows and takes the last round of tiles if it splits it;
                         // grouped_gemm_t_kernel, NT/NN: > 0: places for workgroups, over which the tiles may be split along k
  int pieces;            // grouped_gemm_t_kernel, TN: k pieces per tile
};

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

// ---- 256x256 tiles with ONE wavefront per SIMD: four wavefronts of 128x128 outputs ------------------------------
// The 256 accumulator registers of a wavefront live in AGPRs, and the loop is written slot by slot: after every
// MFMA exactly one LDS or memory instruction (fragment read, staging-register write to LDS, buffer load), so that
// the matrix pipe never waits for a burst of them and the LDS queue never fills.  A 64-deep k slice is loaded
// into registers THREE slices ahead (two staging sets of 16 x 16 bytes per lane), written to the LDS stage that
// is not being read during the first half of a slice, published by the slice's one barrier and read as fragments
// one k step (16) ahead of the MFMAs that use them.  Against eight wavefronts of 128x64 (two per SIMD): a third
// fewer fragment reads per MFMA, and the MFMAs of one wavefront run back to back instead of two wavefronts
// alternating on the pipe.
// Tiles in LDS: k-contiguous operands as [256 rows][64 k] with unpadded 128-byte rows, the 16-byte chunk index
// XORed with (row / 2) % 8 (conflict-free 16-byte row-fragment reads); a k-strided operand (B of the NN product,
// [k][n] row-major) as [64 k][256 n] with 512-byte rows, chunk ^= 4 (k % 4) + (k / 4) % 4 inside each 256-byte
// half row, read as fragments by LDS transpose reads.
//
// The loads are buffer loads issued from assembly: the compiler does not count them, every use of a staging
// register is ordered by a hand-written s_waitcnt vmcnt (loads return in order), and between its load and its
// LDS write a staging register is touched by nothing else (every build checks the generated assembly for this:
// check_grouped_gemm_loops in dhellam_amd/build.py).  The buffer descriptors do the edge handling: their
// length is cut at the group's (or n's) last row, so that rows past the end read as zero and no access leaves
// the operands, whatever the offsets table says.
typedef int gg_i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ gg_i32x4 gg_rsrc(const void *ptr, int64_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)ptr;
  const uint32_t nb = bytes <= 0 ? 0u : (bytes > 0x7fffffffll ? 0x7fffffffu : (uint32_t)bytes);
  gg_i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu));   // stride 0: raw buffer
  r[2] = __builtin_amdgcn_readfirstlane((int)nb);
  r[3] = 0x00020000;
  return r;
}

// Stores a 256x256 tile held in the accumulator layout of grouped_gemm_w4_kernel (wavefront w = 2 wm + wn owns the
// 128x128 block (wm, wn); acc[i][j] is its 32x32 block (i, j), transposed: lane column c is output row c).
template <typename T, bool MAY_ACCUMULATE>
__device__ __forceinline__ void gg_w4_store(const floatx16 (&acc)[4][4], unsigned char *smem, const GGParams &p, T *cbase, int m0,
                                            int n0, int a_rext, int b_rext) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int wm = w >> 1, wn = w & 1;
  // Epilogue: each wavefront passes its 128x128 block through a private LDS region, 64 rows at a time, and stores
  // whole 256-byte row segments (16 lanes a row, 4 rows per instruction).  Rows of 264 bytes: the 8-byte writes of
  // 32 lanes (32 rows, one column) fall on different banks.
  constexpr int EP = 264;
  static_assert(4 * 64 * EP <= 128 * 1024, "epilogue staging fits in the stage buffers");
  unsigned char *ep = smem + w * (64 * EP);
  T *cg = cbase + (int64_t)m0 * p.ldc + n0 + wn * 128;
  struct alignas(8) Q4 { T v[4]; };
  if (MAY_ACCUMULATE && p.accumulate) {
    // c += product with one rounding: straight from the accumulators (a lane owns output row c of each 32x32 block
    // and 4 consecutive columns per register quad)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = wm * 128 + 32 * i + c;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int vb = 0; vb < 4; ++vb) {
          const int n = 32 * j + 8 * vb + 4 * hh;
          if (m < a_rext && wn * 128 + n < b_rext) {
            Q4 *dst = reinterpret_cast<Q4 *>(cg + (int64_t)m * p.ldc + n);
            const Q4 old = *dst;
            Q4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[i][j][4 * vb + e] + static_cast<float>(old.v[e]));
            *dst = o;
          }
        }
    }
    return;
  }
  const int er = lane >> 4, ec = lane & 15;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i2 = 0; i2 < 2; ++i2)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const floatx16 av = acc[2 * h + i2][j];
#pragma unroll
        for (int vb = 0; vb < 4; ++vb) {
          Q4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(av[4 * vb + e]);
          *reinterpret_cast<Q4 *>(ep + (32 * i2 + c) * EP + (32 * j + 8 * vb + 4 * hh) * (int)sizeof(T)) = o;
        }
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int mh = wm * 128 + 64 * h;                   // first row of this half in the tile
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      const int r = 4 * it + er;
      const dh_u32x4 o = *reinterpret_cast<const dh_u32x4 *>(ep + r * EP + ec * 16);
      if (mh + r < a_rext && wn * 128 + 8 * ec < b_rext)
        *reinterpret_cast<dh_u32x4 *>(cg + (int64_t)(mh + r) * p.ldc + 8 * ec) = o;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
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
__global__ void __launch_bounds__(256) grouped_gemm_w4_kernel(const GGParams p) {
  constexpr bool BKS = FORM >= 1, AKS = FORM == 2;
  static_assert(!(AKS && SK), "the wgrad form has many tiles and a short k: it is never split");
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int BM = 256, ROWB = 128, BROWB = 512, TILEB = 256 * ROWB, STAGEB = 2 * TILEB;
  constexpr int NRD = AKS ? 16 : (BKS ? 12 : 8);        // LDS read instructions per k step
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * STAGEB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int wm = w >> 1, wn = w & 1;
  const int nsl = (int)(p.k_dim / 64);
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
        for (int v = tid; v < nv; v += 256) *reinterpret_cast<dh_u32x4 *>(row + 8 * v) = dh_u32x4{0u, 0u, 0u, 0u};
      }
    }
  }

  // ---- copies ----------------------------------------------------------------------------------------------
  // k-contiguous tile [256 rows][64 k]: a lane copies chunk lc of rows lr + 32 i.
  // k-strided tile [64 k][256 n]: a lane copies chunk cx of k rows kr + 8 i.
  const int lc = tid & 7, lr = tid >> 3, cx = tid & 31, kr = tid >> 5;
  const uint32_t goff_a = AKS ? (uint32_t)kr * lda_b + (uint32_t)(cx * 16) : (uint32_t)lr * lda_b + (uint32_t)(lc * 16);
  const uint32_t goff_b = BKS ? (uint32_t)kr * ldb_b + (uint32_t)(cx * 16) : (uint32_t)lr * ldb_b + (uint32_t)(lc * 16);
  const uint32_t kstep_a = AKS ? 64 * lda_b : 64 * (uint32_t)sizeof(T);       // bytes from one k slice to the next
  const uint32_t kstep_b = BKS ? 64 * ldb_b : 64 * (uint32_t)sizeof(T);
  const uint32_t rstep_a = AKS ? 8 * lda_b : 32 * lda_b, rstep_b = BKS ? 8 * ldb_b : 32 * ldb_b;   // bytes from one copy of a lane to its next
  const uint32_t wr_kc = (uint32_t)(lr * ROWB + ((lc ^ ((lr >> 1) & 7)) << 4));                     // + i * 4096
  // k-strided tile: chunk XOR 4 (k % 4) + (k / 4) % 4 with k = kr + 8 i: the i part is bit 1 of the chunk for odd i
  const uint32_t wr_ks = (uint32_t)(kr * BROWB + (cx >> 4) * 256 + (((cx & 15) ^ (4 * (kr & 3) + (kr >> 2))) << 4));
  const uint32_t wr_a = AKS ? wr_ks : wr_kc, wr_b = (uint32_t)TILEB + (BKS ? wr_ks : wr_kc);

  // ---- fragment reads --------------------------------------------------------------------------------------
  const uint32_t sw = (uint32_t)((hh ^ ((c >> 1) & 7)) << 4);
  const uint32_t fa_lane = (uint32_t)((wm * 128 + c) * ROWB) + sw;                  // k step: XOR 32 ks; block i: + 4096 i
  const uint32_t fb_lane = (uint32_t)(TILEB + (wn * 128 + c) * ROWB) + sw;
  const int r16 = lane & 15;
  const int t_lc = 2 * ((lane >> 4) & 1) + ((r16 & 3) >> 1);
  const int tx = 4 * (r16 >> 2) + 2 * hh;
  const uint32_t t_row = (uint32_t)((8 * hh + (r16 >> 2)) * BROWB + ((r16 & 3) & 1) * 8);
  const uint32_t t_lo = t_row + (uint32_t)((t_lc ^ tx) << 4);                       // k rows 8 hh + 0..3 of a step
  const uint32_t t_hi = t_row + 4 * BROWB + (uint32_t)((t_lc ^ (tx + 1)) << 4);     // k rows 8 hh + 4..7
  const uint32_t tb_a = (uint32_t)(TILEB + wn * 256) + t_lo, tb_b = (uint32_t)(TILEB + wn * 256) + t_hi;   // B tile, this wavefront's 128 columns
  const uint32_t ta_a = (uint32_t)(wm * 256) + t_lo, ta_b = (uint32_t)(wm * 256) + t_hi;                   // A tile (TN)
  typedef __attribute__((address_space(3))) const Frag *lds_frag;
  typedef short4v __attribute__((address_space(3))) *lds_tr;
  typedef __attribute__((address_space(3))) gg_i32x4 *lds_w;

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
  // the scalar offset with the length, so a row past the end reads as zero whichever 32-row block it is in.
  // (k-strided operands: cut at the last k row, i.e. the group's last row for TN; in the other direction a tile that
  // reaches past n or m reads what follows in the operand, into outputs that are not stored)
  const gg_i32x4 rsa_ = AKS ? gg_rsrc(ag, (int64_t)(row_end - row_begin) * lda_b - (int64_t)m0 * (int)sizeof(T))
                           : gg_rsrc(ag, (int64_t)(a_rext < 256 ? a_rext : 256) * lda_b);
  const gg_i32x4 rsb_ = AKS ? gg_rsrc(bg, (int64_t)(row_end - row_begin) * ldb_b - (int64_t)n0 * (int)sizeof(T))
                     : BKS ? gg_rsrc(bg, (int64_t)p.k_dim * ldb_b - (int64_t)n0 * (int)sizeof(T))
                           : gg_rsrc(bg, (int64_t)(b_rext < 256 ? b_rext : 256) * ldb_b);
  // The descriptors come out of v_readfirstlane, and a memory instruction may read such a scalar register five wait
  // states later at the earliest.  The compiler keeps that distance for its own instructions, not for the loads issued
  // from assembly below: without this the first of them went out with the previous contents of the length, now and then
  // (a group of fewer than 64 rows then took rows of its neighbour into its weight gradient).
  gg_i32x4 rsa = rsa_, rsb = rsb_;
  asm volatile("s_nop 4" : "+s"(rsa), "+s"(rsb));
  const int cnt = s1 - s0;                              // slices of this segment
  floatx16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  gg_i32x4 stg[2][16];
  Frag fa[2][4];                                        // A fragments, k-contiguous form
  short4v fat[2][4][2];                                 // k-strided form
  Frag fbr[2][4];                                       // B fragments, k-contiguous form
  short4v fbt[2][4][2];                                 // k-strided form: the two transpose reads of a fragment

  auto gload = [&](int set, int idx, uint32_t ka, uint32_t kb) {   // idx 0..7: A, 8..15: B; ka, kb: byte offsets of the slice
    if (idx < 8) asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen" : "=&v"(stg[set][idx]) : "v"(goff_a), "s"(rsa), "s"(ka + idx * rstep_a) : "memory");
    else asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen" : "=&v"(stg[set][idx]) : "v"(goff_b), "s"(rsb), "s"(kb + (idx - 8) * rstep_b) : "memory");
  };
  // kc_w / kc_a / kc_b: the stage's lane addresses for the k-contiguous operands' writes and fragment reads, formed once
  // per slice and kept in registers (left to the compiler they are re-added in front of every LDS instruction)
  auto swrite = [&](int set, int idx, uint32_t stage, uint32_t kc_w) {  // stage: LDS byte address of the stage
    if (idx < 8 && !AKS) *(lds_w)(kc_w + idx * 4096) = stg[set][idx];
    else if (idx < 8) *(lds_w)(((stage + wr_a) ^ (uint32_t)((idx & 1) << 5)) + idx * 4096) = stg[set][idx];
    else if (!BKS) *(lds_w)(kc_w + TILEB + (idx - 8) * 4096) = stg[set][idx];
    else *(lds_w)(((stage + wr_b) ^ (uint32_t)(((idx - 8) & 1) << 5)) + (idx - 8) * 4096) = stg[set][idx];
  };
  // read r of a k step, in the order in which the MFMAs first need the data: B0 A0 B1 B2 B3 A1 A2 A3 (a k-strided
  // B fragment is two transpose reads).  abase/bbase: lane addresses of the stage with the k step applied.
  // a stage's lane addresses for k-contiguous fragment reads, and its base for the k-strided ones
  struct Bases { uint32_t kc_a, kc_b, stage; };
  auto bases_of = [&](uint32_t stage) { return Bases{stage + fa_lane, stage + fb_lane, stage}; };
  auto fread = [&](int set, int r, int ks, const Bases &ba) {
    if constexpr (!BKS) {
      constexpr int isb[8] = {1, 0, 1, 1, 1, 0, 0, 0}, blk[8] = {0, 0, 1, 2, 3, 1, 2, 3};
      if (!isb[r]) fa[set][blk[r]] = *(lds_frag)((ba.kc_a ^ (uint32_t)(ks << 5)) + blk[r] * 4096);
      else fbr[set][blk[r]] = *(lds_frag)((ba.kc_b ^ (uint32_t)(ks << 5)) + blk[r] * 4096);
    } else if constexpr (AKS) {
      // B0 A0 B1 B2 B3 A1 A2 A3, two transpose reads each
      constexpr int isb[8] = {1, 0, 1, 1, 1, 0, 0, 0}, blk[8] = {0, 0, 1, 2, 3, 1, 2, 3};
      const int f = r >> 1, half = r & 1;
      const uint32_t lane_addr = isb[f] ? (half ? tb_b : tb_a) : (half ? ta_b : ta_a);
      const short4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(((ba.stage + lane_addr) ^ (uint32_t)(blk[f] << 6)) + (uint32_t)(ks * 16 * BROWB)));
      if (isb[f]) fbt[set][blk[f]][half] = x;
      else fat[set][blk[f]][half] = x;
    } else {
      constexpr int kind[12] = {1, 2, 0, 1, 2, 1, 2, 1, 2, 0, 0, 0}, blk[12] = {0, 0, 0, 1, 1, 2, 2, 3, 3, 1, 2, 3};
      if (kind[r] == 0) fa[set][blk[r]] = *(lds_frag)((ba.kc_a ^ (uint32_t)(ks << 5)) + blk[r] * 4096);
      else if (kind[r] == 1)
        fbt[set][blk[r]][0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(((ba.stage + tb_a) ^ (uint32_t)(blk[r] << 6)) + (uint32_t)(ks * 16 * BROWB)));
      else
        fbt[set][blk[r]][1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(((ba.stage + tb_b) ^ (uint32_t)(blk[r] << 6)) + (uint32_t)(ks * 16 * BROWB)));
    }
  };

  // prologue: slice 0 into stage 0 (through set 0), slice 1 into set 1, slice 2 into set 0.  Loads of slices that
  // do not exist repeat the last slice (their data is written to a stage nobody reads).
  const int last = cnt > 0 ? cnt - 1 : 0;
  auto kof = [&](int s) { return (uint32_t)(s0 + (s < last ? s : last)); };
#pragma unroll
  for (int x = 0; x < 16; ++x) gload(0, x, kof(0) * kstep_a, kof(0) * kstep_b);
#pragma unroll
  for (int x = 0; x < 16; ++x) gload(1, x, kof(1) * kstep_a, kof(1) * kstep_b);
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
#pragma unroll
  for (int x = 0; x < 16; ++x) swrite(0, x, lds0, lds0 + wr_kc);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  // issue order of a staging set inside the loop: 0..7, 15, 8..14
#pragma unroll
  for (int x = 0; x < 8; ++x) gload(0, x, kof(2) * kstep_a, kof(2) * kstep_b);
  gload(0, 15, kof(2) * kstep_a, kof(2) * kstep_b);
#pragma unroll
  for (int x = 8; x < 15; ++x) gload(0, x, kof(2) * kstep_a, kof(2) * kstep_b);
  asm volatile("s_barrier" ::: "memory");
  {
    const Bases b0 = bases_of(lds0);
#pragma unroll
    for (int x = 0; x < NRD; ++x) fread(0, x, 0, b0);
  }

  // Slice s reads stage s % 2, writes slice s + 1 (staging set (s + 1) % 2, loaded two slices ago) into the other
  // stage during its first half and then loads slice s + 3 into the same set.
  int st = 0;
  auto slice = [&](auto xc, auto lastc, int s) {
    constexpr int X = decltype(xc)::value;              // s % 2
    constexpr bool LAST = decltype(lastc)::value;       // the last slice of an odd count: nothing to prepare
    uint32_t cur = lds0 + (uint32_t)(st * STAGEB), nxt = lds0 + (uint32_t)((st ^ 1) * STAGEB);
    const uint32_t ka = kof(s + 3) * kstep_a, kb = kof(s + 3) * kstep_b;
    asm volatile("" : "+s"(cur), "+s"(nxt));
    Bases bc = bases_of(cur), bn = bases_of(nxt);
    uint32_t wn_ = nxt + wr_kc;
    if constexpr (!AKS) asm volatile("" : "+v"(bc.kc_a), "+v"(bn.kc_a), "+v"(wn_));
    if constexpr (!BKS) asm volatile("" : "+v"(bc.kc_b), "+v"(bn.kc_b));
    // (the k-strided operands' addresses are left to the compiler: pinned, they cost more additions than they save)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mi = 0; mi < 64; ++mi) {
      const int ks = mi >> 4, i = (mi >> 2) & 3, j = mi & 3, q = mi & 15;
      if constexpr (AKS) acc[i][j] = M::mma(frag_join<T>(fbt[ks & 1][j][0], fbt[ks & 1][j][1]), frag_join<T>(fat[ks & 1][i][0], fat[ks & 1][i][1]), acc[i][j]);
      else if constexpr (BKS) acc[i][j] = M::mma(frag_join<T>(fbt[ks & 1][j][0], fbt[ks & 1][j][1]), fa[ks & 1][i], acc[i][j]);
      else acc[i][j] = M::mma(fbr[ks & 1][j], fa[ks & 1][i], acc[i][j]);
      // fragment reads of the next k step, spread over the quarter (the last quarter: behind the barrier, from the next stage)
      if (ks < 3) {
        if (NRD == 8) { if (q % 2 == 0) fread((ks + 1) & 1, q / 2, ks + 1, bc); }
        else if (NRD == 12) { if (q % 4 != 3) fread((ks + 1) & 1, q - q / 4, ks + 1, bc); }
        else fread((ks + 1) & 1, q, ks + 1, bc);
      } else if (!LAST) {
        if (mi == 50) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (NRD == 8) {
          if (mi >= 50 && mi % 2 == 0) fread(0, (mi - 50) / 2, 0, bn);
          if (mi == 63) fread(0, 7, 0, bn);
        } else if (NRD == 12) {
          if (mi >= 50 && mi < 62) fread(0, mi - 50, 0, bn);
        } else {
          if (mi >= 50) fread(0, mi - 50, 0, bn);
          if (mi == 50) fread(0, 14, 0, bn);
          if (mi == 51) fread(0, 15, 0, bn);
        }
      }
      if (!LAST && mi < 32 && mi % 2 == 1) {            // LDS writes of slice s + 1: the older of the two sets in flight
        const int k = mi / 2;
        if (k == 0) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
        if (k == 8) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        swrite(X ^ 1, k, nxt, wn_);
      }
      if (!LAST && mi >= 33 && mi <= 61 && mi % 2 == 1) gload(X ^ 1, (mi - 33) / 2, ka, kb);
      if (!LAST && mi == 48) gload(X ^ 1, 15, ka, kb);
      __builtin_amdgcn_sched_barrier(0);
    }
    st ^= 1;
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  int s = 0;
#pragma unroll 1
  for (; s + 1 < cnt; s += 2) {
    slice(I0{}, std::false_type{}, s);
    slice(I1{}, std::false_type{}, s + 1);
  }
  // The loads of the last slices (unused data) still target the staging registers: wait for them, and keep the
  // registers reserved until then (for the compiler a load whose result nobody reads frees its register at once).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int x = 0; x < 16; ++x) asm volatile("" ::"v"(stg[0][x]), "v"(stg[1][x]));
  if (s < cnt) slice(I0{}, std::true_type{}, s);
  __syncthreads();                                      // everyone is done with the stages: they stage the output below

  if constexpr (SK) {
    // 16 bytes per lane and instruction: piece ((w * 16 + i * 4 + j) * 4 + vb) of the tile, 1 KB each
    float *dst = part + ((size_t)w * 64 * 4 + 0) * 64 + (size_t)lane * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int vb = 0; vb < 4; ++vb) {
          const floatx16 av = acc[i][j];
          const floatx4 o = {av[4 * vb], av[4 * vb + 1], av[4 * vb + 2], av[4 * vb + 3]};
          *reinterpret_cast<floatx4 *>(dst + (size_t)(((i * 4 + j) * 4 + vb) * 256)) = o;
        }
    __syncthreads();                                    // the next segment's copies reuse the stages
    return;
  }
  gg_w4_store<T, AKS>(acc, smem, p, AKS ? reinterpret_cast<T *>(p.c) + (int64_t)g * p.c_group_stride : reinterpret_cast<T *>(p.c), m0, n0, a_rext, b_rext);
    __syncthreads();                                    // the next segment's copies reuse the staging area
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
  } else if constexpr (!SK) {
    // The grid is sized for the host's upper bound of the tile count (it does not know how the rows split into
    // groups); the chunks of the XCDs are cut from the real count, so that every XCD gets its share of real tiles.
    int tiles_m;
    const GGGroupTable gt = gg_group_table(p, base, tiles_m);
    const int ntiles = tiles_m * p.tiles_n;
    int kept = ntiles;
    if (p.sk_grid > 0) {
      // the tiles past the last full round of sk_grid tiles belong to the split kernel, if it splits them
      const int full = ntiles / p.sk_grid, rem = ntiles - full * p.sk_grid;
      if (gg_sk_pieces(p.sk_grid, rem, nsl) > 1) kept = full * p.sk_grid;
    }
    if ((int)blockIdx.x >= kept) return;
    const int pid = gg_xcd_chunk((int)blockIdx.x, kept);              // (the XCDs share the tiles that are computed here)
    int tm_all, tn, g, rb, re, tm;
    gg_tile_of(pid, tiles_m, p.tiles_n, tm_all, tn);
    gg_locate(gt, tm_all, g, rb, re, tm);
    segment(g, rb, re, tm, tn, 0, nsl, nullptr);
  } else {
    // The last round of tiles, split along k.  The tiles (in the order of gg_tile_of) run in rounds of gridDim.x = the
    // number of compute units; grouped_gemm_w4_kernel<.., false> in front of this kernel takes the full rounds, one
    // workgroup per tile.  When the last round holds at most half as many tiles as there are workgroups, it is left to
    // this kernel: as many k pieces per tile as fit (workgroup w: tile w % rem, piece w / rem, so that neighbours work
    // on neighbouring tiles), summed afterwards in k order.  288 tiles on 256 compute units then take 1 1/8 tile
    // times instead of 2.  (A resident workgroup that also looped over the full rounds was 3-6 % slower on them than
    // one workgroup per tile.)
    int tiles_m;
    const GGGroupTable gt = gg_group_table(p, base, tiles_m);
    const int tiles = tiles_m * p.tiles_n;
    const int grid = (int)gridDim.x, full = tiles / grid, rem = tiles - full * grid;
    const int pieces = gg_sk_pieces(grid, rem, nsl);
    const int wg = gg_xcd_chunk((int)blockIdx.x, grid);                // neighbouring tiles on one XCD
    if (pieces == 1 || wg >= rem * pieces) return;
    const int ts = wg % rem, pc = wg / rem;
    int tm_all, tn, g, rb, re, tm;
    gg_tile_of(full * grid + ts, tiles_m, p.tiles_n, tm_all, tn);
    gg_locate(gt, tm_all, g, rb, re, tm);
    segment(g, rb, re, tm, tn, pc * nsl / pieces, (pc + 1) * nsl / pieces, p.ws + (size_t)wg * (256 * 256));
  }
}

// Sums the k pieces of the tiles of a split last round, in k order (deterministic), and stores the tiles.
// 16 workgroups per tile of that round: a wavefront takes one 32x32 block (w, i, j) of the accumulator layout,
// reads its 4 KB of every piece (1 KB per instruction) and writes 4 columns per lane and register quad.
template <typename T>
__global__ void __launch_bounds__(256) gg_split_reduce_kernel(const GGParams p, int sk_grid) {
  constexpr int BM = 256;
  const int nsl = (int)(p.k_dim / 64);
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
  const int blk = (blockIdx.x % 16) * 4 + (tid >> 6);   // (w * 4 + i) * 4 + j
  const int w = blk >> 4, i = (blk >> 2) & 3, j = blk & 3;
  floatx4 acc[4];
#pragma unroll
  for (int vb = 0; vb < 4; ++vb) acc[vb] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int pc = 0; pc < pieces; ++pc) {
    const float *src = p.ws + (size_t)(pc * rem + ts) * (256 * 256) + (size_t)blk * (4 * 256) + (size_t)lane * 4;
#pragma unroll
    for (int vb = 0; vb < 4; ++vb) acc[vb] += *reinterpret_cast<const floatx4 *>(src + vb * 256);
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
  const int c = lane & 31, hh = lane >> 5;
  const int m = (w >> 1) * 128 + 32 * i + c, n = (w & 1) * 128 + 32 * j + 4 * hh;    // + 8 vb
  const int m0 = rb + tm * BM, n0 = tn * 256;
  if (m0 + m >= re) return;
  T *dst = reinterpret_cast<T *>(p.c) + (int64_t)(m0 + m) * p.ldc + n0 + n;
  struct alignas(8) Q4 { T v[4]; };
#pragma unroll
  for (int vb = 0; vb < 4; ++vb)
    if (n0 + n + 8 * vb < p.n_dim) {
      Q4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[vb][e]);
      *reinterpret_cast<Q4 *>(dst + 8 * vb) = o;
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
// LDS: a k-contiguous operand as [rows][64 k] (128-byte rows, 16-byte chunk XOR (row / 2) % 8), a k-strided one as
// [64 k][128 columns] (256-byte rows, chunk XOR 4 (k % 4) + (k / 4) % 4), as in grouped_gemm_w4_kernel; a wavefront
// copies 1 KB per instruction, so the XOR is applied to the global chunk that a lane fetches.  Buffer descriptors cut
// the operands at the group's last row (k-strided: last k row), past which a copy writes zeros; columns past n read
// what follows in the same operand and end in outputs that are not stored.
template <typename T>
__device__ __forceinline__ void gg_copy_lds(uint32_t lane_off, const gg_i32x4 &rsrc, uint32_t off, uint32_t lds_dst) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(lane_off), "s"(rsrc), "s"(off), "s"(lds_dst)
               : "memory", "m0");
}

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

template <int FORM, int BM, int BN> struct GGT {
  static constexpr bool AKS = FORM == 2, BKS = FORM >= 1;
  static constexpr int NW = BN / 32;                            // wavefronts
  static constexpr int WM = BM == 32 ? 1 : 2, WN = NW / WM;     // over the tile
  static constexpr int MI = BM / (32 * WM), NI = BN / (32 * WN); // 32x32 blocks of a wavefront
  static constexpr int NST = BN == 256 ? 3 : BM == 128 ? 2 : BM == 64 ? 3 : 4;  // stages: 144 KB; 64, 72, 80 KB
  static constexpr int ABYTES = BM * 128, STAGE = ABYTES + BN * 128;
  static constexpr int ACPW = BM / (8 * NW), BCPW = BN / (8 * NW), CPW = ACPW + BCPW;   // copies of a wavefront per slice
  static constexpr int PER_CU = BN == 256 ? 1 : 2;              // workgroups that share a compute unit
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

template <typename T, int FORM, int BM, int BN>
__global__ void __launch_bounds__(2 * BN, 2) grouped_gemm_t_kernel(const GGParams p) {
  using C = GGT<FORM, BM, BN>;
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr bool AKS = C::AKS, BKS = C::BKS;
  constexpr int MI = C::MI, NI = C::NI;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[C::NST * C::STAGE];
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
  gg_i32x4 ra, rb;
  auto descriptors = [&](int s) {
    ra = gg_rsrc(ag + s * kstep_a, a_len - s * kstep_a);
    rb = gg_rsrc(bg + s * kstep_b, b_len - s * kstep_b);
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
      gg_copy_lds<T>(v, ra, (uint32_t)((AKS ? 4 : 8) * b) * lda_b, stage + (uint32_t)(b * 1024));
    } else {
      const int y = x - C::ACPW, b = w * C::BCPW + y;             // (a k-strided B tile of 256 columns is two of 128)
      uint32_t v = vb[y];
      if (!BKS && tail) {
        const int ch = ((lane & 7) ^ (lane >> 4)) ^ (4 * (b & 1));
        if (ch * 8 >= kc_tail) v = OUT;
      }
      const uint32_t off = BKS ? (uint32_t)(4 * (b & 15)) * ldb_b + (uint32_t)((b >> 4) * 256) : (uint32_t)(8 * b) * ldb_b;
      gg_copy_lds<T>(v, rb, off, stage + (uint32_t)(C::ABYTES + b * 1024));
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
    if (MORE || s + C::NST - 2 < cnt) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((C::NST - 2) * C::CPW) : "memory");
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
#pragma unroll 1
  for (; s + C::NST - 1 < cnt; ++s) slice(std::true_type{}, s);
#pragma unroll 1
  for (; s < cnt; ++s) slice(std::false_type{}, s);

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
  constexpr int EP = NI * 64 + 8, LPR = NI * 4;                   // region row in bytes, lanes per row of 16-byte pieces
  static_assert(C::NW * 32 * MI * EP <= C::NST * C::STAGE, "staging fits in the stages");
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
static int launch_gg_w4_tn(GGParams p, hipStream_t st) {
  p.tiles_m = (int)cdiv(p.m_dim, 256);
  p.tiles_n = (int)cdiv(p.n_dim, 256);
  hipLaunchKernelGGL((grouped_gemm_w4_kernel<T, 2, false>), dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.groups), dim3(256), 0, st, p);
  return DH_OK;
}

template <typename T, bool BKS>
static int launch_gg_w4(GGParams p, int64_t m_extent, void *workspace, size_t workspace_bytes, hipStream_t st) {
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
  // known): the first kernel then leaves that round to the split kernel.  When nothing is split the two extra
  // launches cost a few microseconds; a split saves up to half a tile time (45 us and more).
  p.sk_grid = grid;
  hipLaunchKernelGGL((grouped_gemm_w4_kernel<T, BKS ? 1 : 0, false>), dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(256), 0, st, p);
  if (grid > 0) {
    p.ws = reinterpret_cast<float *>(workspace);
    p.zero_tail = 0;                                    // done by the kernel above
    hipLaunchKernelGGL((grouped_gemm_w4_kernel<T, BKS ? 1 : 0, true>), dim3((unsigned)grid), dim3(256), 0, st, p);
    hipLaunchKernelGGL((gg_split_reduce_kernel<T>), dim3((unsigned)(16 * grid / 2)), dim3(256), 0, st, p, grid);   // at most grid / 2 tiles are split
  }
  return DH_OK;
}

template <typename T, int FORM, int BM, int BN>
static int launch_gg_t(GGParams p, int64_t m_extent, void *workspace, size_t workspace_bytes, hipStream_t st) {
  using C = GGT<FORM, BM, BN>;
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
  hipLaunchKernelGGL((grouped_gemm_t_kernel<T, FORM, BM, BN>), dim3((unsigned)grid), dim3(2 * BN), 0, st, p);
  if (reduce > 0)
    hipLaunchKernelGGL((gg_t_reduce_kernel<T, FORM, BM, BN>), dim3((unsigned)cdiv(reduce * BLOCKS, 4)), dim3(256), 0, st, p);
  return DH_OK;
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
    return launch_gg_t<T, FORM, 128, 128>(p, m_extent, workspace, workspace_bytes, st);
  }
}

// NT / NN: whether 256x256 tiles, one workgroup per compute unit, are the faster ones: enough of them, and a reduction long
// enough to pay for their start and end (6036 rows of 4 groups, n = 7168 of 4096: 326 us against 380 us in 128x256 tiles;
// 16384 rows of 8 groups, n = 4096 of 704: 53 against 37 us in 128x128 tiles).
static bool gg_w4_pays(int64_t rows, int64_t n, int64_t k) {
  const int64_t tiles = cdiv(rows, 256) * cdiv(n, 256);
  return tiles >= 256 && (k >= 1536 || (k >= 640 && tiles >= 1500));
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
  const bool big = gg_w4_pays(max_rows, n, k);
  if (big && k % 64 == 0 && k <= (1ll << 21)) {
    rc = dtype == DH_BF16 ? launch_gg_w4<bf16_t, false>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : launch_gg_w4<f16_t, false>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
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
  const bool big = gg_w4_pays(max_rows, n, k);
  if (big && k % 64 == 0 && k <= (1ll << 21) && k * n * (int64_t)dtype_size(dtype) < (1ll << 31)) {
    rc = dtype == DH_BF16 ? launch_gg_w4<bf16_t, true>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream)
                          : launch_gg_w4<f16_t, true>(p, max_rows, workspace, workspace_bytes, (hipStream_t)stream);
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
  // 256x256 tiles where the groups have many rows and there is much to do altogether (6000 rows of 8 groups, 7168 x 2048:
  // 200 against 228 us in 128x128 tiles; 20000 rows of 16 groups, 2816 x 512: 77 against 70 us); their offsets have to fit
  // the 32-bit buffer addressing
  if (max_rows / groups >= 384 && cdiv(m, 256) * cdiv(n, 256) * max_rows >= 600000 &&
      max_rows * (m > n ? m : n) * (int64_t)dtype_size(dtype) < (1ll << 31))
    rc = dtype == DH_BF16 ? launch_gg_w4_tn<bf16_t>(p, (hipStream_t)stream) : launch_gg_w4_tn<f16_t>(p, (hipStream_t)stream);
  else
    rc = dtype == DH_BF16 ? dispatch_gg_t<bf16_t, 2>(p, m, workspace, workspace_bytes, (hipStream_t)stream)
                          : dispatch_gg_t<f16_t, 2>(p, m, workspace, workspace_bytes, (hipStream_t)stream);
  if (rc) return rc;
  DH_LAUNCH_CHECK();
  return DH_OK;
}

extern "C" int dh_grouped_gemm_tn(const void *a, const void *b, void *c, const int32_t *offs, int groups,
                                  int64_t max_rows, int64_t m, int64_t n, int accumulate, int dtype, void *stream) {
  return dh_grouped_gemm_tn_ws(a, b, c, offs, groups, max_rows, m, n, accumulate, dtype, nullptr, 0, stream);
}
