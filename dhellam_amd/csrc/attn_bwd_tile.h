// Attention backward on the tile layout of attn_tile.h (16 bits), two passes: dQ (which forms delta = rowsum(dO O) and runs
// first) and dK/dV, or both in one grid behind a delta kernel.  Workgroup shape and what bounds it: as the forward kernel
// (attn_fwd_tile.h).
// dK/dV keeps K and V fragments and both accumulators in registers (196 at head dim 64, 244 at 96): two wavefronts a SIMD, one
// at the larger head dims (332 at 128; at 256 all 512 and 75 more that are spilled, 216 bytes a lane).  dQ at head dim 128
// in its 64-row form spills 8 of 256, outside the loop.
// Measured, backward, causal, register-staged kernels / these with a memory latency exposed in every iteration / now: 16 heads x
// 2 x 512, head dim 64 58 / 24 / 22 us; 32 query / 8 kv heads x 4096, head dim 64 1313 / 326 / 290, 96 1562 / 440 / 420, 256 10871 / 1842
// / 1736 us; 16 heads x 1024, head dim 192 - / 95 / 82 us.
#include "attn_tile.h"

namespace dh {

// dQ: RG row groups of 32 query rows x SPLIT splits of the keys, 32-key tiles of K and V.
template <int D, int RG, int SPLIT> constexpr int dq_tile_lds() {
  const int all = 2 * SPLIT * 2 * 32 * D * 2, ex = (SPLIT - 1) * RG * 32 * D * 4;
  return all > ex ? all : ex;
}
// Workgroup bx of gx of sequence by of gy; DELTA: it forms delta, else delta is there already.
template <typename T, int D, int RG, int SPLIT, bool DELTA>
__device__ __forceinline__ void dq_tile_body(const AttnBwdParams &p, int bx, int gx, int by, int gy, char *sAll, float *sDel) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int BM = 32 * RG, BN = 32, NW = RG * SPLIT, SLOTF = 32 * D;
  constexpr int TILEB = BN * D * (int)sizeof(T);
  constexpr int STAGEB = SPLIT * 2 * TILEB;
  static_assert(sizeof(T) == 2, "dq_tile_lds");
  constexpr int RPW = SPLIT * 2 * BN / NW;                // rows that a wavefront copies per iteration
  static_assert(RPW % 16 == 0 && RPW <= BN, "whole copy patterns of one tile per wavefront");

  const int b = seq_by_length(p.cu_q, gy, by);
  const int ratio = p.hq / p.hk, P = gx / p.hq;
  int hkv, item;
  xcd_group_item(bx, p.hk, ratio * P, hkv, item);
  const int h = hkv * ratio + item % ratio, px = item / ratio;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nqt = (sq + BM - 1) / BM;
  if constexpr (DELTA) delta_tail_zero<BM>(p, b, h, sq, px);
  if (px >= nqt) return;
  const int m0 = (nqt - 1 - px) * BM;          // late causal tiles carry the most work and come first
  const int causal = p.causal;
  const float scale_log2 = p.scale_log2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int rg = w % RG, sp = w / RG;
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;

  // copies of this wavefront: rows cp_r0 .. + RPW - 1 of the K or V tile of split cp_sp
  constexpr int PARTS = BN / RPW;
  const int cp_r0 = RPW * (w % PARTS), cp_v = (w / PARTS) & 1, cp_sp = w / (2 * PARTS);
  const int64_t cp_stride = cp_v ? p.v_stride : p.k_stride;
  const T *cp_g = reinterpret_cast<const T *>(cp_v ? p.v : p.k) + (int64_t)k0 * cp_stride + (int64_t)hkv * D;
  const TileCopy<D> cl = tile_copy<D>(lane, (uint32_t)(cp_stride * (int64_t)sizeof(T)));
  const int cp_whole = tile_whole_rows(sk, cp_stride);
  const uint32_t cp_dst = lds0 + (uint32_t)(cp_v * SPLIT * TILEB + cp_sp * TILEB + cp_r0 * D * (int)sizeof(T));

  int nk_end = sk;
  if (causal && m0 + BM < nk_end) nk_end = m0 + BM;
  const int ntiles = (nk_end + BN - 1) / BN;
  const int niter = (ntiles + SPLIT - 1) / SPLIT;
  auto issue = [&](int it) {
    const int tile = it * SPLIT + cp_sp;
    if (tile < ntiles) copy_tile<T, D, RPW>(cp_g, cp_stride, tile * BN + cp_r0, sk, cp_whole, cp_dst + (uint32_t)((it & 1) * STAGEB), cl, lane);
  };
  if (niter > 0) issue(0);

  const int wrow0 = m0 + rg * 32, row_q = wrow0 + c;
  const bool row_ok = row_q < sq;
  const int row_ld = row_ok ? row_q : sq - 1;
  Frag Qf[D / 16], dOf[D / 16];
  {
    const T *qp = reinterpret_cast<const T *>(p.q) + (int64_t)(q0 + row_ld) * p.q_stride + (int64_t)h * D + 8 * hh;
    const T *dp = reinterpret_cast<const T *>(p.dout) + (int64_t)(q0 + row_ld) * p.do_stride + (int64_t)h * D + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      Qf[ks] = frag_ld<T>(qp + ks * 16);
      dOf[ks] = frag_ld<T>(dp + ks * 16);
    }
  }
  const int64_t stat = ((int64_t)b * p.hq + h) * p.max_sq + row_q;
  const float lse_c = row_ok ? p.lse[((int64_t)b * p.hq + h) * p.lse_pitch + row_q] * 1.4426950408889634f : INFINITY;        // rows past the end: P = 0
  float del_c = 0.f;
  if (!DELTA) {
    if (row_ok) del_c = p.delta[stat];
  } else if (sp == 0) {       // delta of the workgroup's rows, for the other splits and for the dK/dV pass
    const T *op = reinterpret_cast<const T *>(p.out) + (int64_t)(q0 + row_ld) * p.o_stride + (int64_t)h * D + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const Frag of = frag_ld<T>(op + ks * 16);
#pragma unroll
      for (int j = 0; j < 8; ++j) del_c += to_f(dOf[ks][j]) * to_f(of[j]);
    }
    del_c = row_ok ? pair32_sum(del_c) : 0.f;
    if (hh == 0) {
      sDel[rg * 32 + c] = del_c;
      if (row_ok) p.delta[stat] = del_c;
      if (row_q < p.ld2_pitch) {          // both, side by side, in whole 32-row tiles (padding rows: zeros)
        const int64_t a2 = ((int64_t)b * p.hq + h) * p.ld2_pitch + row_q;
        p.ld2[a2] = row_ok ? lse_c : 0.f;
        p.ld2[p.ld2_plane + a2] = -del_c;
      }
    }
  }
  const RowLane rl = row_lane<D>(lane);
  const TrLane tl = tr_lane<D>(lane);

  floatx16 dQt[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) dQt[t][v] = 0.f;
  if constexpr (DELTA) {
    __syncthreads();
    del_c = sDel[rg * 32 + c];
  }

  loaded_here(Qf);
  loaded_here(dOf);
  float stats[2] = {lse_c, del_c};
  loaded_here(stats);
#pragma unroll 1
  for (int it = 0; it < niter; ++it) {
    dma_wait_all();
    __syncthreads();                             // this stage has landed, and everyone is done with the other one
    if (it + 1 < niter) issue(it + 1);
    const int tile = it * SPLIT + sp, n0 = tile * BN;
    if (tile < ntiles && !(causal && n0 > wrow0 + 31)) {
      const uint32_t kt = lds0 + (uint32_t)((it & 1) * STAGEB + sp * TILEB);
      floatx16 S, dP;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        S[v] = 0.f;
        dP[v] = 0.f;
      }
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        S = M::mma(row_frag<T, D>(kt, rl, ks), Qf[ks], S);
        dP = M::mma(row_frag<T, D>(kt + (uint32_t)(SPLIT * TILEB), rl, ks), dOf[ks], dP);
      }
      if ((causal && n0 + BN - 1 > wrow0) || n0 + BN > sk) {
        const int lim = causal && row_q + 1 < sk ? row_q + 1 : sk;
#pragma unroll
        for (int v = 0; v < 16; ++v) S[v] = n0 + acc_row(v, hh) < lim ? S[v] : -INFINITY;        // P = dS = 0
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float ds[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) ds[j] = fast_exp2(S[8 * s + j] * scale_log2 - stats[0]) * (dP[8 * s + j] - stats[1]);
        const Frag dSb = frag_pack<T>(ds);
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
          dQt[t] = M::mma(tr_frag<T, D>(kt, tl, t, s), dSb, dQt[t]);
      }
    }
  }
  __syncthreads();

  // add the splits' partial dQ through LDS, in split order: slot x = (split - 1) * RG + row group
  float *xo = reinterpret_cast<float *>(sAll);
  if (sp > 0) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) xo[((sp - 1) * RG + rg) * SLOTF + (t * 16 + v) * 64 + lane] = dQt[t][v];
  }
  __syncthreads();
  if (sp > 0 || !row_ok) return;
#pragma unroll
  for (int s2 = 1; s2 < SPLIT; ++s2)
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) dQt[t][v] += xo[((s2 - 1) * RG + rg) * SLOTF + (t * 16 + v) * 64 + lane];
  T *dqp = reinterpret_cast<T *>(p.dq) + (int64_t)(q0 + row_q) * p.dq_stride + (int64_t)h * D;
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int vb = 0; vb < 4; ++vb) {
      Quad<T> *at = reinterpret_cast<Quad<T> *>(dqp + 32 * t + 8 * vb + 4 * hh), a;
      if (p.dq_accumulate) a = *at;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        a.v[e] = static_cast<T>((p.dq_accumulate ? static_cast<float>(a.v[e]) : 0.f) + dQt[t][4 * vb + e] * p.scale);
      *at = a;
    }
}

template <typename T, int D, int RG, int SPLIT, int WPS>
__global__ void __launch_bounds__(64 * RG * SPLIT, WPS) attn_bwd_dq_tile_kernel(const AttnBwdParams p) {
  __shared__ __attribute__((aligned(1024))) char sAll[dq_tile_lds<D, RG, SPLIT>()];
  __shared__ float sDel[32 * RG];
  dq_tile_body<T, D, RG, SPLIT, true>(p, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y, sAll, sDel);
}

// dK, dV: KG row groups of 32 key rows x QSPLIT splits of the query tiles (32 rows of Q and dO each); K and V row
// fragments stay in registers; lse and delta of a tile, from the planes that the kernel before it wrote, are copied along
// with it (256 bytes each, of which the first 128 count).
template <int D, int QSPLIT> constexpr int dkv_tile_stage() { return QSPLIT * (2 * 32 * D * 2 + 512); }
template <int D, int QSPLIT> constexpr int dkv_tile_lds() {
  return 2 * dkv_tile_stage<D, QSPLIT>();
}
template <typename T, int D, int KG, int QSPLIT>
__device__ __forceinline__ void dkv_tile_body(const AttnBwdParams &p, int bx, int gx, int by, int gy, char *sAll) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int BN = 32 * KG, BM = 32, NW = KG * QSPLIT, SLOTF = 32 * D;
  constexpr int TILEB = BM * D * (int)sizeof(T);          // bytes of one Q (or dO) tile
  constexpr int STAGEB = dkv_tile_stage<D, QSPLIT>();     // per split: Q tile, dO tile; behind them, per split: lse, delta
  static_assert(sizeof(T) == 2, "dkv_tile_stage");
  static_assert(QSPLIT * 2 == NW, "one whole tile per wavefront");

  const int b = seq_by_length(p.cu_k, gy, by);
  const int G = p.hk * p.hsplit;
  int hg, px;
  xcd_group_item(bx, G, gx / G, hg, px);
  const int hkv = hg / p.hsplit, hs = hg % p.hsplit;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int j0 = px * BN;          // early causal tiles carry the most work and come first
  if (j0 >= sk) return;
  const int causal = p.causal;
  const float scale_log2 = p.scale_log2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int kg = w % KG, qs = w / KG;
  const int ratio = p.hq / p.hk, hper = ratio / p.hsplit;
  const int h_first = hkv * ratio + hs * hper;
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;
  const int jw0 = j0 + 32 * kg, jrow = jw0 + c;

  // copies of this wavefront: the Q (even) or dO (odd) tile of split w / 2
  const int cp_do = w & 1, cp_sp = w >> 1;
  const int64_t cp_stride = cp_do ? p.do_stride : p.q_stride;
  const T *cp_g = reinterpret_cast<const T *>(cp_do ? p.dout : p.q) + (int64_t)q0 * cp_stride;
  const TileCopy<D> cl = tile_copy<D>(lane, (uint32_t)(cp_stride * (int64_t)sizeof(T)));
  const int cp_whole = tile_whole_rows(sq, cp_stride);
  const uint32_t cp_dst = lds0 + (uint32_t)((cp_sp * 2 + cp_do) * TILEB);

  const int i_begin = causal ? j0 : 0;
  const int ntq = i_begin < sq ? (sq - i_begin + BM - 1) / BM : 0;
  const int it_per_head = (ntq + QSPLIT - 1) / QSPLIT;
  const int niter = it_per_head * hper;
  int gi = 0, si = 0;                                     // head and step of the next iteration to be copied
  const float *ld_g = p.ld2 + (cp_do ? p.ld2_plane : 0) + c;
  auto issue = [&](int slot) {
    const int tq = si * QSPLIT + cp_sp, row0 = i_begin + tq * BM;
    if (tq < ntq) {
      copy_tile<T, D, BM>(cp_g + (int64_t)(h_first + gi) * D, cp_stride, row0, sq, cp_whole, cp_dst + (uint32_t)(slot * STAGEB), cl, lane);
      const float *src = ld_g + ((int64_t)b * p.hq + (h_first + gi)) * p.ld2_pitch + row0;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
                   : : "v"(src), "s"(lds0 + (uint32_t)(slot * STAGEB + QSPLIT * 2 * TILEB + (cp_sp * 2 + cp_do) * 256)) : "memory", "m0");
    }
    if (++si == it_per_head) { si = 0; ++gi; }
  };
  if (niter > 0) issue(0);

  Frag Kf[D / 16], Vf[D / 16];
  {
    const int jl = jrow < sk ? jrow : sk - 1;
    const T *kp = reinterpret_cast<const T *>(p.k) + (int64_t)(k0 + jl) * p.k_stride + (int64_t)hkv * D + 8 * hh;
    const T *vp = reinterpret_cast<const T *>(p.v) + (int64_t)(k0 + jl) * p.v_stride + (int64_t)hkv * D + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      Kf[ks] = frag_ld<T>(kp + ks * 16);
      Vf[ks] = frag_ld<T>(vp + ks * 16);
    }
  }
  floatx16 dKt[D / 32], dVt[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      dKt[t][v] = 0.f;
      dVt[t][v] = 0.f;
    }
  const RowLane rl = row_lane<D>(lane);
  const TrLane tl = tr_lane<D>(lane);
  loaded_here(Kf);
  loaded_here(Vf);
  int ti = 0;                                             // step of iteration it
#pragma unroll 1
  for (int it = 0; it < niter; ++it) {
    dma_wait_all();
    __syncthreads();                                      // this stage has landed, and everyone is done with the other one
    if (it + 1 < niter) issue((it + 1) & 1);
    const int tq = ti * QSPLIT + qs, i0 = i_begin + tq * BM;
    if (tq < ntq && !(causal && i0 + BM - 1 < jw0)) {
      const uint32_t qt = lds0 + (uint32_t)((it & 1) * STAGEB + qs * 2 * TILEB), dt = qt + (uint32_t)TILEB;
      // lse (exp2 units) and delta of the rows 8 vb + 4 hh + e
      typedef __attribute__((address_space(3))) const floatx4 *lds_f4;
      const uint32_t lt = lds0 + (uint32_t)((it & 1) * STAGEB + QSPLIT * 2 * TILEB + qs * 512 + 16 * hh);
      floatx4 l4[4], d4[4];
#pragma unroll
      for (int vb = 0; vb < 4; ++vb) {
        l4[vb] = *(lds_f4)(lt + 32 * vb);
        d4[vb] = *(lds_f4)(lt + 256 + 32 * vb);
      }
      floatx16 S, dP;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        S[v] = 0.f;
        dP[v] = 0.f;
      }
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        S = M::mma(row_frag<T, D>(qt, rl, ks), Kf[ks], S);
        dP = M::mma(row_frag<T, D>(dt, rl, ks), Vf[ks], dP);
      }
      if ((causal && i0 < jw0 + 31) || i0 + BM > sq) {
        const int lo = causal ? jrow : 0;           // first query row that attends to this lane's key
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int i = i0 + acc_row(v, hh);
          S[v] = i >= lo && i < sq ? S[v] : -INFINITY;        // P = dS = 0
        }
      }
      Frag Pb[2], dSb[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float pv[8], dsv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int v = 8 * s + j;
          pv[j] = fast_exp2(S[v] * scale_log2 - l4[v >> 2][v & 3]);
          dsv[j] = pv[j] * (dP[v] + d4[v >> 2][v & 3]);      // (the plane holds -delta)
        }
        Pb[s] = frag_pack<T>(pv);
        dSb[s] = frag_pack<T>(dsv);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < D / 32; ++t) {
          dVt[t] = M::mma(tr_frag<T, D>(dt, tl, t, s), Pb[s], dVt[t]);
          dKt[t] = M::mma(tr_frag<T, D>(qt, tl, t, s), dSb[s], dKt[t]);
        }
    }
    if (++ti == it_per_head) ti = 0;
  }
  __syncthreads();

  // add the splits' partial sums through LDS in a fixed order, halving: (0 += 2, 1 += 3), then 0 += 1; per (split, key
  // group): dK, then dV
  static_assert(2 * STAGEB >= (QSPLIT / 2) * KG * 2 * SLOTF * 4, "exchange area");
  float *xo = reinterpret_cast<float *>(sAll);
#pragma unroll
  for (int from = QSPLIT / 2; from >= 1; from >>= 1) {
    if (qs >= from && qs < 2 * from) {
      float *dst = xo + ((qs - from) * KG + kg) * (2 * SLOTF) + lane;
#pragma unroll
      for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          dst[(t * 16 + v) * 64] = dKt[t][v];
          dst[SLOTF + (t * 16 + v) * 64] = dVt[t][v];
        }
    }
    __syncthreads();
    if (qs < from) {
      const float *src = xo + (qs * KG + kg) * (2 * SLOTF) + lane;
#pragma unroll
      for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          dKt[t][v] += src[(t * 16 + v) * 64];
          dVt[t][v] += src[SLOTF + (t * 16 + v) * 64];
        }
    }
    __syncthreads();
  }
  if (qs > 0 || jrow >= sk) return;
  if (p.hsplit == 1) {
    T *dkp = reinterpret_cast<T *>(p.dk) + (int64_t)(k0 + jrow) * p.dk_stride + (int64_t)hkv * D;
    T *dvp = reinterpret_cast<T *>(p.dv) + (int64_t)(k0 + jrow) * p.dv_stride + (int64_t)hkv * D;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int vb = 0; vb < 4; ++vb) {
        Quad<T> a, bq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a.v[e] = static_cast<T>(dKt[t][4 * vb + e] * p.scale);
          bq.v[e] = static_cast<T>(dVt[t][4 * vb + e]);
        }
        *reinterpret_cast<Quad<T> *>(dkp + 32 * t + 8 * vb + 4 * hh) = a;
        *reinterpret_cast<Quad<T> *>(dvp + 32 * t + 8 * vb + 4 * hh) = bq;
      }
  } else {
    const int64_t off = (((int64_t)hs * p.total_k + (k0 + jrow)) * p.hk + hkv) * D;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int vb = 0; vb < 4; ++vb) {
        floatx4 a, bq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] = dKt[t][4 * vb + e] * p.scale;
          bq[e] = dVt[t][4 * vb + e];
        }
        *reinterpret_cast<floatx4 *>(p.dk_part + off + 32 * t + 8 * vb + 4 * hh) = a;
        *reinterpret_cast<floatx4 *>(p.dv_part + off + 32 * t + 8 * vb + 4 * hh) = bq;
      }
  }
}

template <typename T, int D, int KG, int QSPLIT, int WPS>
__global__ void __launch_bounds__(64 * KG * QSPLIT, WPS) attn_bwd_dkv_tile_kernel(const AttnBwdParams p) {
  __shared__ __attribute__((aligned(1024))) char sAll[dkv_tile_lds<D, QSPLIT>()];
  dkv_tile_body<T, D, KG, QSPLIT>(p, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y, sAll);
}

// delta, with the lse / delta planes, in front of the two passes in one launch: two lanes a row, which add in the order of the
// dQ kernel's prologue.  (Where all of a sequence's attention is on one key, dS is the difference of two roundings: in another
// order dQ and dK would be other noise.)
template <typename T, int D> __global__ void __launch_bounds__(256) attn_bwd_delta_kernel(const AttnBwdParams p) {
  const int b = blockIdx.y, q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0, hh = threadIdx.x & 1;
  const int rows = p.delta_tail ? p.max_sq : sq, padded = (sq + 31) / 32 * 32, all = rows > padded ? rows : padded;
  for (int64_t item = (int64_t)blockIdx.x * 128 + (threadIdx.x >> 1); item < (int64_t)all * p.hq; item += (int64_t)gridDim.x * 128) {
    const int i = (int)(item / p.hq), h = (int)(item % p.hq);
    float s = 0.f;
    if (i < sq) {
      const T *dp = reinterpret_cast<const T *>(p.dout) + (int64_t)(q0 + i) * p.do_stride + (int64_t)h * D + 8 * hh;
      const T *op = reinterpret_cast<const T *>(p.out) + (int64_t)(q0 + i) * p.o_stride + (int64_t)h * D + 8 * hh;
      typename Mma<T>::Frag df[D / 16], of[D / 16];
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        df[ks] = frag_ld<T>(dp + ks * 16);
        of[ks] = frag_ld<T>(op + ks * 16);
      }
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) s += to_f(df[ks][j]) * to_f(of[ks][j]);
    }
    s += __shfl_xor(s, 1, 64);                   // both lanes of a row are at the same item
    const int64_t head = (int64_t)b * p.hq + h;
    if (hh == 0 && i < rows) p.delta[head * p.max_sq + i] = s;
    if (i < padded) p.ld2[(hh ? p.ld2_plane : 0) + head * p.ld2_pitch + i] = hh ? -s : i < sq ? p.lse[head * p.lse_pitch + i] * 1.4426950408889634f : 0.f;
  }
}

// Both passes in one launch, behind the delta kernel: ndkv workgroups a sequence do dK/dV and, after those of all sequences,
// ndq a sequence dQ.
template <typename T, int D, int RG, int SPLIT, int KG, int QSPLIT, int WPS>
__global__ void __launch_bounds__(64 * RG * SPLIT, WPS) attn_bwd_both_tile_kernel(const AttnBwdParams p, int ndkv, int ndq, int batch) {
  static_assert(RG * SPLIT == KG * QSPLIT, "one workgroup shape");
  constexpr int A = dq_tile_lds<D, RG, SPLIT>(), B = dkv_tile_lds<D, QSPLIT>();
  __shared__ __attribute__((aligned(1024))) char sAll[A > B ? A : B];
  const int i = blockIdx.x, j = i - ndkv * batch;
  if (j < 0) dkv_tile_body<T, D, KG, QSPLIT>(p, i % ndkv, ndkv, i / ndkv, batch, sAll);
  else dq_tile_body<T, D, RG, SPLIT, false>(p, j % ndq, ndq, j / ndq, batch, sAll, nullptr);
}

template <typename T, int D, int RG, int SPLIT, int WPS>
static int launch_dq_tile(const AttnBwdParams &p, int batch, hipStream_t st) {
  dim3 grid((unsigned)(cdiv(p.max_sq, 32 * RG) * p.hq), (unsigned)batch);
  hipLaunchKernelGGL((attn_bwd_dq_tile_kernel<T, D, RG, SPLIT, WPS>), grid, dim3(64 * RG * SPLIT), 0, st, p);
  return DH_OK;
}

template <typename T, int D, int KG, int QSPLIT, int WPS>
static int launch_dkv_tile(const AttnBwdParams &p, int batch, int max_sk, hipStream_t st) {
  dim3 grid((unsigned)(cdiv(max_sk, 32 * KG) * p.hk * p.hsplit), (unsigned)batch);
  hipLaunchKernelGGL((attn_bwd_dkv_tile_kernel<T, D, KG, QSPLIT, WPS>), grid, dim3(64 * KG * QSPLIT), 0, st, p);
  return DH_OK;
}

template <typename T, int D, int RG, int SPLIT, int KG, int QSPLIT, int WPS>
static int launch_both_tile(const AttnBwdParams &p, int batch, int max_sk, hipStream_t st) {
  const int64_t items = (int64_t)p.ld2_pitch * p.hq, blocks = cdiv(items, 128) < 4096 ? cdiv(items, 128) : 4096;
  hipLaunchKernelGGL((attn_bwd_delta_kernel<T, D>), dim3((unsigned)blocks, (unsigned)batch), dim3(256), 0, st, p);
  const int64_t ndkv = cdiv(max_sk, 32 * KG) * p.hk * p.hsplit, ndq = cdiv(p.max_sq, 32 * RG) * p.hq;
  hipLaunchKernelGGL((attn_bwd_both_tile_kernel<T, D, RG, SPLIT, KG, QSPLIT, WPS>), dim3((unsigned)((ndkv + ndq) * batch)),
                     dim3(64 * RG * SPLIT), 0, st, p, (int)ndkv, (int)ndq, batch);
  return DH_OK;
}

}  // namespace dh
