// dQ from recomputed S and dP at head dim 128 in 16 bits: one wavefront on a SIMD, every instruction of the main loop in a fixed order.
#pragma once
#include "attn_loops.inc"
#include "attn_rows.h"

namespace dh {

// A workgroup is RG row groups x 4 / RG key splits (4 x 1 or 2 x 2): a wavefront holds 64 query rows (Q and dO: 128 registers, dQ: 128)
// and walks its split's tiles of 32 keys.  The wavefronts of a split share its tiles and copy them together, three ahead; loop and
// meeting point are attn_loops.py's.  S^T = K Q^T and dP^T = V dO^T - delta have the query index on lanes, so that P and dS need
// one lse and one delta a lane and dS^T is the operand of dQ^T += K^T dS^T as it is: 112 vector instructions, 32 LDS reads and 8 copies
// for 96 MFMAs.  The prologue forms delta = rowsum(dO O), writes it and the planes that dK/dV reads: this kernel runs before it.
// Two splits' partial sums go through LDS; each adds up and stores half of the rows.  Causal: row tiles i and n - 1 - i.
// What it measured: 1860 cycles a tile (two splits 1915 for two), of which the matrix pipe is busy 1536, and 15000 and 16500 cycles to load and
// store a tile's rows; the eight wavefronts 3400 and 9000.  32 query / 8 kv heads, causal 4096 210 -> 166 us, 4096 rows x 2048 keys 213 -> 166, seven
// packed sequences of 1 to 3324 tokens 283 -> 234.  Key blocks that no row of a block of 32 sees get no products: a key that is not finite reaches
// dQ of the rows in its block and behind, no further.
template <typename T, int RG>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) attn_bwd_dq128_kernel(const AttnBwdParams p) {
  constexpr int D = 128, BM = 64 * RG, BN = 32, SPLIT = 4 / RG, STAGES = 4;
  constexpr int COPIES = 16 / RG, CROWS = 4 * COPIES;  // 1 KB copies of a wavefront a tile, and their rows
  constexpr uint32_t ROWB = 2 * D, TILEB = BN * ROWB, STAGEB = 2 * TILEB, STREAMB = STAGES * STAGEB;
  // the tiles; behind them (and, with two splits, in the stages that are filled last) 16 KB a wavefront for its own rows
  constexpr uint32_t OWN = 64 * ROWB, LDS = SPLIT * STREAMB + (RG == 4 ? 4 : 2) * OWN;
  static_assert(OWN == STAGEB && (SPLIT == 1 || SPLIT * STREAMB == 4 * 32768), "own rows, exchange area");
  __shared__ __attribute__((aligned(1024))) char sAll[LDS];

  if (p.delta_tail) {
    const int y = blockIdx.y, rows = (p.cu_q[y + 1] >> p.q_shift) - (p.cu_q[y] >> p.q_shift);
    if (rows < p.max_sq) {
      const int tiles = (p.max_sq + BM - 1) / BM, P = p.causal ? (tiles + 1) / 2 : tiles, head = blockIdx.x / P, x = blockIdx.x - head * P;
      delta_tail_zero<BM>(p, y, head, rows, x);
      if (p.causal && tiles - 1 - x != x) delta_tail_zero<BM>(p, y, head, rows, tiles - 1 - x);
    }
  }
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
  const int rg = w % RG, sp = w / RG;
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;
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
    const int ntiles = (nk_end + BN - 1) / BN;
    int rem = (ntiles + SPLIT - 1) / SPLIT;           // tiles of each split; those past the end are masked

    uint32_t cl[4];
    rows_lanes(cl, lane, c_rowb);
    int key = sp * BN;
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st) {
      const int row = (sp + SPLIT * st) * BN, rows = sk - crow - row < CROWS ? sk - crow - row : CROWS;
      const int4v rs = rows_rsrc(c_base + (int64_t)row * c_rowb, rows > 0 ? (uint32_t)(rows - 1) * c_rowb + ROWB : 0u);
#pragma unroll
      for (int i = 0; i < COPIES; ++i) copy_1k(cl[i & 3], rs, i < 4 ? 0u : c16, cdst + st * STAGEB + 1024u * i);
    }
    const int next = (sp + SPLIT * (STAGES - 1)) * BN, left = sk - crow - next;
    const char *cp = c_base + (int64_t)next * c_rowb;
    const int64_t cstep = (int64_t)SPLIT * BN * c_rowb;

    int4v Q[4][4], dO[4][4];                          // query block, k step
    floatx4 nd[4];
    float lse[4], del[4];
    {
      // rows of Q, dO and O through LDS, a KB a copy (gathered from memory, 16 rows of 64 bytes a load, the three took 18000 to 25000
      // cycles of a tile's rows)
      const uint32_t own = lds0 + (RG == 4 ? STREAMB + (uint32_t)w * OWN : w < 2 ? (uint32_t)w * STREAMB + 3 * STAGEB : 2 * STREAMB + (uint32_t)(w - 2) * OWN);
      typedef __attribute__((address_space(3))) const int4v *lds_i4;
      const int rows = sq - wrow0 < 64 ? sq - wrow0 : 64;
      auto fetch = [&](const void *base, int64_t stride, int4v (&f)[4][4]) {
        const uint32_t rowb = (uint32_t)stride * 2u;
        uint32_t off[4];
        rows_lanes(off, lane, rowb);
        const int4v rs = rows_rsrc(reinterpret_cast<const T *>(base) + (int64_t)(q0 + wrow0) * stride + (int64_t)h * D, rows > 0 ? (uint32_t)(rows - 1) * rowb + ROWB : 0u);
#pragma unroll
        for (int i = 0; i < 16; ++i) copy_1k(off[i & 3], rs, (uint32_t)(i >> 2) * 16u * rowb, own + 1024u * i);
        dma_wait_all();
#pragma unroll
        for (int qb = 0; qb < 4; ++qb)
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) f[qb][ks] = *(lds_i4)(own + (uint32_t)(qb * 4096 + r * 256) + ((uint32_t)((4 * ks + g) ^ swz16(r)) << 4));
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) loaded_here(f[qb]);      // read, before anything else is copied there
      };
#pragma unroll
      for (int qb = 0; qb < 4; ++qb) {
        const int row = wrow0 + 16 * qb + r;
        lse[qb] = p.lse[((int64_t)b * p.hq + h) * p.lse_pitch + (row < sq ? row : sq - 1)];
      }
      int4v O[4][4];
      fetch(p.q, p.q_stride, Q);
      fetch(p.dout, p.do_stride, dO);
      fetch(p.out, p.o_stride, O);
#pragma unroll
      for (int qb = 0; qb < 4; ++qb) {
        del[qb] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const auto of = __builtin_bit_cast(typename Mma<T>::Frag, O[qb][ks]), df = __builtin_bit_cast(typename Mma<T>::Frag, dO[qb][ks]);
#pragma unroll
          for (int j = 0; j < 8; ++j) del[qb] += to_f(df[j]) * to_f(of[j]);
        }
        del[qb] += __shfl_xor(del[qb], 16, 64);
        del[qb] += __shfl_xor(del[qb], 32, 64);
        const bool ok = wrow0 + 16 * qb + r < sq;
        if (!ok) del[qb] = 0.f;
        lse[qb] = ok ? lse[qb] * 1.4426950408889634f : INFINITY;
        nd[qb] = floatx4{-del[qb], -del[qb], -del[qb], -del[qb]};
      }
    }
    if (sp == 0 && g == 0) {                          // also with the copy that dK/dV streams (zeros in the rows that pad a tile)
#pragma unroll
      for (int qb = 0; qb < 4; ++qb) {
        const int row = wrow0 + 16 * qb + r;
        if (row < sq) p.delta[((int64_t)b * p.hq + h) * p.max_sq + row] = del[qb];
        if (row < p.ld2_pitch) {
          const int64_t a2 = ((int64_t)b * p.hq + h) * p.ld2_pitch + row;
          p.ld2[a2] = row < sq ? lse[qb] : 0.f;
          p.ld2[p.ld2_plane + a2] = -del[qb];
        }
      }
    }
    // fragment reads: row r, chunk 4 ks + g; transposed: rows 4 g + r / 4 (and 16 further), chunk 2 t + (r % 4) / 2
    uint32_t rk[4], ta[8];
    {
      const uint32_t row = stream + (uint32_t)(r * ROWB), x = (uint32_t)((g ^ swz16(r)) << 4);
#pragma unroll
      for (uint32_t ks = 0; ks < 4; ++ks) rk[ks] = row + (x ^ (ks << 6));
      const int tr = 4 * g + (r >> 2), ch = (r & 3) >> 1;
      const uint32_t at = stream + (uint32_t)(tr * ROWB + 8 * (r & 1));
#pragma unroll
      for (int t = 0; t < 8; ++t) ta[t] = at + (uint32_t)(((ch ^ swz16(tr)) ^ (2 * t)) << 4);
    }
    const int vx = causal ? 4 * g - r - wrow0 : -(1 << 30), vy = 4 * g - sk;      // key - row and key - keys, but for the tile's first key
    // tiles from this key on have something to mask
    const int mlim = causal && wrow0 - BN + 1 < sk - BN ? wrow0 - BN + 1 : sk - BN;
    const int alim = causal ? wrow0 + 31 : 1 << 30;   // ... and past this key lie behind the first 32 rows
    floatx4 o[4][8];                                  // query block, d block
#define DH_ACC4(qb, t) [o##qb##t] "=&a"(o[qb][t])
#define DH_ACC(qb) \
  DH_ACC4(qb, 0), DH_ACC4(qb, 1), DH_ACC4(qb, 2), DH_ACC4(qb, 3), DH_ACC4(qb, 4), DH_ACC4(qb, 5), DH_ACC4(qb, 6), DH_ACC4(qb, 7)
#define DH_ROW(x, X, qb) [x##qb##0] "a"(X[qb][0]), [x##qb##1] "a"(X[qb][1]), [x##qb##2] "a"(X[qb][2]), [x##qb##3] "a"(X[qb][3])
#define DH_LOOP(TEXT)                                                                                                                \
  asm volatile(TEXT                                                                                                                 \
               : DH_ACC(0), DH_ACC(1), DH_ACC(2), DH_ACC(3), [rem] "+s"(rem)                                                         \
               : DH_ROW(q, Q, 0), DH_ROW(q, Q, 1), DH_ROW(q, Q, 2), DH_ROW(q, Q, 3), DH_ROW(d, dO, 0), DH_ROW(d, dO, 1),             \
                 DH_ROW(d, dO, 2), DH_ROW(d, dO, 3), [rk0] "v"(rk[0]), [rk1] "v"(rk[1]), [rk2] "v"(rk[2]), [rk3] "v"(rk[3]),          \
                 [ta0] "v"(ta[0]), [ta1] "v"(ta[1]), [ta2] "v"(ta[2]), [ta3] "v"(ta[3]), [ta4] "v"(ta[4]), [ta5] "v"(ta[5]),          \
                 [ta6] "v"(ta[6]), [ta7] "v"(ta[7]), [cl0] "v"(cl[0]), [cl1] "v"(cl[1]), [cl2] "v"(cl[2]), [cl3] "v"(cl[3]),          \
                 [lse0] "v"(lse[0]), [lse1] "v"(lse[1]), [lse2] "v"(lse[2]), [lse3] "v"(lse[3]), [nd0] "v"(nd[0]), [nd1] "v"(nd[1]),  \
                 [nd2] "v"(nd[2]), [nd3] "v"(nd[3]), [vx] "v"(vx), [vy] "v"(vy), [scale] "s"(p.scale_log2), [cp] "s"(cp),             \
                 [cstep] "s"(cstep), [left] "s"(left), [key] "s"(key), [keystep] "s"(SPLIT * BN), [crowb] "s"(c_rowb), [c16] "s"(c16), \
                 [cdst] "s"(cdst), [mlim] "s"(mlim), [alim] "s"(alim)                                                                                 \
               : DH_DQ128_CLOBBERS)
    if constexpr (__is_same(T, bf16_t)) {
      if constexpr (COPIES == 4) DH_LOOP(DH_DQ128_LOOP_BF16_4);
      else DH_LOOP(DH_DQ128_LOOP_BF16_8);
    } else {
      if constexpr (COPIES == 4) DH_LOOP(DH_DQ128_LOOP_F16_4);
      else DH_LOOP(DH_DQ128_LOOP_F16_8);
    }
#undef DH_LOOP
#undef DH_ROW
#undef DH_ACC
#undef DH_ACC4
    __syncthreads();                                  // everyone is done with the tiles
    auto store = [&](int qb, const floatx4 (&sum)[8]) {
      const int row = wrow0 + 16 * qb + r;
      if (row >= sq) return;
      struct alignas(8) Four { T v[4]; };
      T *dqp = reinterpret_cast<T *>(p.dq) + (int64_t)(q0 + row) * p.dq_stride + (int64_t)h * D + 4 * g;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        Four *dst = reinterpret_cast<Four *>(dqp + 16 * t), a;
        if (p.dq_accumulate) {
          a = *dst;
#pragma unroll
          for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(static_cast<float>(a.v[e]) + sum[t][e] * p.scale);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(sum[t][e] * p.scale);
        }
        *dst = a;
      }
    };
    if constexpr (SPLIT == 1) {
#pragma unroll
      for (int qb = 0; qb < 4; ++qb) store(qb, o[qb]);
    } else {
      // split sp takes the query blocks 2 sp, 2 sp + 1 of its row group: split 0's part + split 1's
      typedef __attribute__((address_space(3))) floatx4 *lds_f4;
      auto block = [&](int split, int qb) { return (lds_f4)(lds0 + (uint32_t)((split * RG + rg) * 32768 + qb * 8192)) + lane; };
#pragma unroll
      for (int qb = 0; qb < 4; ++qb) {
        const lds_f4 dst = block(sp, qb);
#pragma unroll
        for (int t = 0; t < 8; ++t) dst[64 * t] = o[qb][t];
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const lds_f4 s0 = block(0, 2 * sp + x), s1 = block(1, 2 * sp + x);
        floatx4 sum[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) sum[t] = s0[64 * t] + s1[64 * t];
        store(2 * sp + x, sum);
      }
      __syncthreads();
    }
  }
}

}  // namespace dh
