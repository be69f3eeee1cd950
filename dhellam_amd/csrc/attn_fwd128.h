// Forward at head dim 128 in 16 bits: one wavefront on a SIMD, every instruction of the main loop in a fixed order.
#pragma once
#include "attn_loops.inc"
#include "attn_rows.h"

namespace dh {

// A workgroup is RG row groups x 4 / RG key splits (4 x 1 or 2 x 2): a wavefront holds 64 query rows (Q: 64 registers, O: 128) and walks
// its split's tiles of 32 keys.  The wavefronts of a split share its tiles and copy them together, three ahead; loop and meeting
// point are attn_loops.py's.  S^T = K Q^T has the query index on lanes, so that P^T
// is the operand of O^T += V^T P^T as it is, and the reference m of the exponentials and the sums l are one a lane and block.
// Whether m has to move is asked of the sum of a lane's eight values, which is needed anyway, instead of their maximum: 112
// vector instructions and four comparisons, 24 LDS reads and 4 copies for 68 MFMAs.
// What it measured: 1740 cycles a tile, of which the matrix pipe is busy 1088: a wavefront issues an instruction in 5 cycles, and there are
// about 290 (barrier 85, the two branches 75).  32 query / 8 kv heads, 4096 rows x 2048 keys 157 -> 129 us (1.07 PFLOP/s), causal
// 4096 156 -> 133, seven packed sequences of 1 to 3324 tokens 215 -> 184.  Errors of out against 64 bits, the eight wavefronts / here: narrow scores
// (queries and keys of variance 1) a little larger, since fewer rows have their largest P at exactly 1 (bf16 causal 4096 2.087e-3 / 2.096e-3, fp16
// 2.606e-4 / 2.617e-4, 32 heads x 600 in 128-row tiles 2.282e-3 / 2.311e-3), scores three and eight times as wide smaller (2.103e-3 / 1.940e-3,
// 1.809e-3 / 1.703e-3).  Without the sums of rounded P and with the first tile as the reference 2.12e-3 where it is 2.09e-3, and 5 % faster.
// O goes through LDS (the loop writes it there) and out in whole rows.  (Q through LDS as well, into the half that the tiles leave free, brought
// nothing: packed sequences 1.256 times the eight wavefronts against 1.255 to 1.268.)  Causal: row tiles i and n - 1 - i.
template <typename T, int RG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) attn_fwd128_kernel(const AttnFwdParams p) {
  constexpr int D = 128, BM = 64 * RG, BN = 32, SPLIT = 4 / RG, STAGES = 4;
  constexpr int COPIES = 16 / RG, CROWS = 4 * COPIES;  // 1 KB copies of a wavefront a tile, and their rows
  constexpr uint32_t ROWB = 2 * D, TILEB = BN * ROWB, STAGEB = 2 * TILEB, STREAMB = STAGES * STAGEB, OUTB = 64 * D * 4;
  static_assert(SPLIT * STREAMB <= 4 * OUTB, "the tiles lie where O is written at the end");
  __shared__ __attribute__((aligned(1024))) char sAll[4 * OUTB];
  __shared__ float sM[4][64], sN[4][64], sL[4][64];    // of each row: reference, sum of P as rounded and sum of P
  rng_state_zero(p);

  const RowWork work = row_work<BM>(p.cu_q, p.q_shift, p.max_sq, p.hq, p.hk, p.causal);
  if (work.b < 0) return;
  const int b = __builtin_amdgcn_readfirstlane(work.b), h = __builtin_amdgcn_readfirstlane(work.h), px = __builtin_amdgcn_readfirstlane(work.px);
  const int hkv = __builtin_amdgcn_readfirstlane(work.hkv);
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nqt = (sq + BM - 1) / BM;
  const int causal = p.causal;
  int qt0 = px, qt1 = 0, nq = 1;
  if (causal) {
    qt0 = nqt - 1 - px; qt1 = px;
    nq = qt0 == qt1 ? 1 : 2;
  }
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;
  const int rg = w % RG, sp = w / RG;
  const uint32_t stream = lds0 + (uint32_t)sp * STREAMB;
  // what this wavefront copies: K (the first half of the row groups) or V, with four groups rows 0..15 or 16..31 of a tile
  const bool copy_v = rg >= RG / 2;
  const int crow = RG == 4 ? 16 * (rg & 1) : 0;
  const int64_t c_stride = copy_v ? p.v_stride : p.k_stride;
  const uint32_t c_rowb = (uint32_t)c_stride * 2u, c16 = 16u * c_rowb;
  const char *c_base = reinterpret_cast<const char *>(reinterpret_cast<const T *>(copy_v ? p.v : p.k) + (int64_t)(k0 + crow) * c_stride + (int64_t)hkv * D);
  const uint32_t cdst = stream + (copy_v ? TILEB : 0u) + (uint32_t)crow * ROWB;

  for (int qi = 0; qi < nq; ++qi) {
    const int m0 = (qi == 0 ? qt0 : qt1) * BM, wrow0 = m0 + 64 * rg;
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));                    // lane addresses are formed anew for each tile of rows
    const int r = lane & 15, g = lane >> 4;
    int nk_end = sk;
    if (causal && m0 + BM < nk_end) nk_end = m0 + BM;
    int rem = ((nk_end + BN - 1) / BN + SPLIT - 1) / SPLIT;      // tiles of each split; those past the end are masked

    uint32_t cl[4];
    rows_lanes(cl, lane, c_rowb);
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st) {
      const int row = (sp + SPLIT * st) * BN, rows = sk - crow - row < CROWS ? sk - crow - row : CROWS;
      const int4v rs = rows_rsrc(c_base + (int64_t)row * c_rowb, rows > 0 ? (uint32_t)(rows - 1) * c_rowb + ROWB : 0u);
#pragma unroll
      for (int i = 0; i < COPIES; ++i) copy_1k(cl[i & 3], rs, i < 4 ? 0u : c16, cdst + st * STAGEB + 1024u * i);
    }
    const int next = (sp + SPLIT * (STAGES - 2)) * BN;      // the loop moves on before it copies
    const int left = sk - crow - next;
    const char *cp = c_base + (int64_t)next * c_rowb;
    const int64_t cstep = (int64_t)SPLIT * BN * c_rowb;

    int4v Q[4][4];                                    // query block, k step
#pragma unroll
    for (int qb = 0; qb < 4; ++qb) {
      const int row = wrow0 + 16 * qb + r, row_ld = row < sq ? row : sq - 1;
      const T *qp = reinterpret_cast<const T *>(p.q) + (int64_t)(q0 + row_ld) * p.q_stride + (int64_t)h * D + 8 * g;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) Q[qb][ks] = *reinterpret_cast<const int4v *>(qp + 32 * ks);
    }
    // fragment reads: row r, chunk 4 ks + g; transposed: rows 4 g + r / 4 (and 16 further), chunk 2 t + (r % 4) / 2; O: row r, 16-byte
    // chunk 4 t + g of 32
    uint32_t rk[4], ta[8], wo[8];
    {
      const uint32_t row = stream + (uint32_t)(r * ROWB), x = (uint32_t)((g ^ swz16(r)) << 4);
#pragma unroll
      for (uint32_t ks = 0; ks < 4; ++ks) rk[ks] = row + (x ^ (ks << 6));
      const int tr = 4 * g + (r >> 2), ch = (r & 3) >> 1;
      const uint32_t at = stream + (uint32_t)(tr * ROWB + 8 * (r & 1));
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        ta[t] = at + (uint32_t)(((ch ^ swz16(tr)) ^ (2 * t)) << 4);
        wo[t] = lds0 + (uint32_t)w * OUTB + (uint32_t)(r * 512 + (((4 * t + g) ^ r) << 4));
      }
    }
    const int vx = causal ? 4 * g - r - wrow0 : -(1 << 30), vy = 4 * g - sk;      // key - row and key - keys, but for the tile's first key
    // tiles from this key on have something to mask
    const int mlim = causal && wrow0 - BN + 1 < sk - BN ? wrow0 - BN + 1 : sk - BN;
    const int alim = causal ? wrow0 + 31 : 1 << 30;   // ... and past this key lie behind the first 32 rows
    float m[4] = {-1e30f, -1e30f, -1e30f, -1e30f}, l[4] = {0.f, 0.f, 0.f, 0.f}, n[4];
#define DH_ROW(x, X, qb) [x##qb##0] "a"(X[qb][0]), [x##qb##1] "a"(X[qb][1]), [x##qb##2] "a"(X[qb][2]), [x##qb##3] "a"(X[qb][3])
#define DH_LOOP(TEXT)                                                                                                                \
  asm volatile(TEXT                                                                                                                 \
               : [m0] "+v"(m[0]), [m1] "+v"(m[1]), [m2] "+v"(m[2]), [m3] "+v"(m[3]), [l0] "+v"(l[0]), [l1] "+v"(l[1]),                \
                 [l2] "+v"(l[2]), [l3] "+v"(l[3]), [n0] "=&v"(n[0]), [n1] "=&v"(n[1]), [n2] "=&v"(n[2]), [n3] "=&v"(n[3]),            \
                 [rem] "+s"(rem)                                                                                                     \
               : DH_ROW(q, Q, 0), DH_ROW(q, Q, 1), DH_ROW(q, Q, 2), DH_ROW(q, Q, 3), [rk0] "v"(rk[0]), [rk1] "v"(rk[1]),              \
                 [rk2] "v"(rk[2]), [rk3] "v"(rk[3]), [ta0] "v"(ta[0]), [ta1] "v"(ta[1]), [ta2] "v"(ta[2]), [ta3] "v"(ta[3]),          \
                 [ta4] "v"(ta[4]), [ta5] "v"(ta[5]), [ta6] "v"(ta[6]), [ta7] "v"(ta[7]), [cl0] "v"(cl[0]), [cl1] "v"(cl[1]),          \
                 [cl2] "v"(cl[2]), [cl3] "v"(cl[3]), [wo0] "v"(wo[0]), [wo1] "v"(wo[1]), [wo2] "v"(wo[2]), [wo3] "v"(wo[3]),          \
                 [wo4] "v"(wo[4]), [wo5] "v"(wo[5]), [wo6] "v"(wo[6]), [wo7] "v"(wo[7]), [vx] "v"(vx), [vy] "v"(vy),                  \
                 [scale] "s"(p.scale_log2), [cp] "s"(cp), [cstep] "s"(cstep), [left] "s"(left), [key] "s"(sp * BN),                   \
                 [keystep] "s"(SPLIT * BN), [crowb] "s"(c_rowb), [c16] "s"(c16), [cdst] "s"(cdst), [mlim] "s"(mlim), [alim] "s"(alim)                  \
               : DH_FWD128_CLOBBERS)
    if constexpr (__is_same(T, bf16_t)) {
      if constexpr (COPIES == 4) DH_LOOP(DH_FWD128_LOOP_BF16_4);
      else DH_LOOP(DH_FWD128_LOOP_BF16_8);
    } else {
      if constexpr (COPIES == 4) DH_LOOP(DH_FWD128_LOOP_F16_4);
      else DH_LOOP(DH_FWD128_LOOP_F16_8);
    }
#undef DH_LOOP
#undef DH_ROW
#pragma unroll
    for (int qb = 0; qb < 4; ++qb) {
      float lt = l[qb];
      lt += __shfl_xor(lt, 16, 64);
      lt += __shfl_xor(lt, 32, 64);
      if (g == 0) {
        sM[w][16 * qb + r] = m[qb];
        sN[w][16 * qb + r] = n[qb];
        sL[w][16 * qb + r] = lt;
      }
    }
    if constexpr (SPLIT > 1) __syncthreads();         // (of one split a wavefront reads what it wrote itself)
    // rows 64 / SPLIT sp .. of the row group: the splits' parts on one reference, in split order, and out in whole rows
    typedef __attribute__((address_space(3))) const floatx4 *lds_f4;
    constexpr int ROWS = 64 / SPLIT;
    const int u = lane & 15;
    T *op = reinterpret_cast<T *>(p.o) + (int64_t)(q0 + wrow0) * p.o_stride + (int64_t)h * D + 8 * u;
#pragma unroll 4
    for (int i = 0; i < ROWS / 4; ++i) {
      const int row = ROWS * sp + 4 * i + (lane >> 4);
      float mx = sM[rg][row];
#pragma unroll
      for (int x = 1; x < SPLIT; ++x) mx = fmaxf(mx, sM[rg + RG * x][row]);
      floatx4 a, c;
      float nt = 0.f, lt = 0.f;
#pragma unroll
      for (int x = 0; x < SPLIT; ++x) {
        const int y = rg + RG * x;
        const uint32_t at = lds0 + (uint32_t)y * OUTB + (uint32_t)(row * 512);
        const floatx4 ax = *(lds_f4)(at + (uint32_t)(((2 * u) ^ (row & 15)) << 4)), cx = *(lds_f4)(at + (uint32_t)(((2 * u + 1) ^ (row & 15)) << 4));
        if constexpr (SPLIT == 1) {
          a = ax, c = cx, nt = sN[y][row], lt = sL[y][row];
        } else {
          const float f = fast_exp2(sM[y][row] - mx);
          a = x == 0 ? ax * f : a + ax * f;
          c = x == 0 ? cx * f : c + cx * f;
          nt += sN[y][row] * f;
          lt += sL[y][row] * f;
        }
      }
      const float inv = nt > 0.f ? 1.0f / nt : 0.f;
      struct alignas(8) Four { T v[4]; } lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo.v[e] = static_cast<T>(a[e] * inv);
        hi.v[e] = static_cast<T>(c[e] * inv);
      }
      if (wrow0 + row < sq) {                         // (rows of O are 8-byte aligned)
        *reinterpret_cast<Four *>(op + (int64_t)row * p.o_stride) = lo;
        *reinterpret_cast<Four *>(op + (int64_t)row * p.o_stride + 4) = hi;
        if (u == 0) p.lse[((int64_t)b * p.hq + h) * p.max_sq + wrow0 + row] = lt > 0.f ? mx * 0.6931471805599453f + logf(lt) : -INFINITY;
      }
    }
    __syncthreads();                                  // the next rows' tiles are copied to where O was
  }
}

}  // namespace dh
