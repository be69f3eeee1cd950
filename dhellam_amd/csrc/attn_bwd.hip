// Flash-attention backward on bf16/fp16 MFMA (gfx950), deterministic (no
// floating-point atomics).
//
// Three kernels (head dim 128 has them in attn_bwd_dkv128.h and attn_bwd_dq128.h, one wavefront on a SIMD):
//   delta   : delta_i = sum_d dO[i,d] * O[i,d]                      (streaming; for fp32 and where dS is kept: the
//             recomputing dQ kernels form delta in their prologue and run first)
//   dK/dV   : a workgroup owns 64 key/value rows (K, V fragments stay in
//             registers, for head dim 128 K in LDS), walks the
//             query heads of its GQA group and the query tiles that attend to
//             it; S = Q K^T and dP = dO V^T are computed
//             with the key index on lanes so that P and dS feed dV^T += dO^T P
//             and dK^T += Q^T dS straight from their accumulators, with the
//             transposed Q / dO fragments coming from LDS transpose reads.
//             The GQA group sum happens in the accumulators; when the grid
//             would be too small the group is split over workgroups and a small
//             kernel adds the fp32 partials in a fixed order.
//   dQ      : a workgroup owns 32*NW query rows (Q, dO fragments in registers),
//             walks the key tiles; S^T, dP^T have the query index on lanes and
//             dS^T feeds dQ^T += K^T dS^T.
// Recomputing S and dP in both passes costs 7 matrix products instead of 5 but
// needs no fp32 dQ accumulator in memory and no atomics.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "attn_route.h"
#include "mma.h"


namespace dh {

struct AttnBwdParams {
  const void *dout, *q, *k, *v;
  const void *out;           // forward output (the dQ kernels form delta from it)
  int64_t o_stride;
  const float *lse;
  float *delta;              // fp32 [batch][hq][max_sq]: rowsum(dO * O); written by the delta kernel or by the dQ kernel
  float *ld2;                // fp32 [2][plane]: lse * log2(e), then -delta, each [batch][hq][ld2_pitch]
  int64_t ld2_plane;         // elements between the two planes
  int ld2_pitch;             // max_sq rounded up to 32: every 32-row query tile of a head is one aligned 128-byte run
  void *dq, *dk, *dv;
  float *dk_part, *dv_part;  // fp32 [hsplit][total_k][hk][d] when hsplit > 1
  const int32_t *cu_q, *cu_k;
  int max_sq, hq, hk, hsplit;
  int64_t total_k;
  int64_t q_stride, k_stride, v_stride, do_stride, dq_stride, dk_stride, dv_stride;
  float scale, scale_log2;
  int causal;
  int q_shift, k_shift;      // sequence bounds are cu >> shift (the halves of a context-parallel chunk)
  int lse_pitch;             // rows of a head in lse
  int dq_accumulate;         // dq += this call's gradient (read, add in fp32, round once) instead of dq =
  int delta_tail;            // delta is an output: its rows past a sequence's end, up to max_sq, are zeros
  // dS = P * (dP - delta) kept for the dQ product (head dim 128, 16 bits, when the workspace allows): 2 KB blocks of
  // 32 keys x 32 query rows, block (b, h, query tile, key block); inside a block the 16-byte piece (s, hh, key)
  // holds the query rows 16 s + 8 u + 4 hh + x of that key (u = 0, 1; x = 0..3): what a lane of the dK/dV kernel
  // has in its packed dS fragment s.
  void *ds;
  int ds_nqt, ds_nkb;        // query tiles and key blocks (of 32) per (batch, head)
};

// Zeros in the rows of delta past the end of the sequence, in tile `tile` of BM rows of the grid laid out for max_sq.  A
// filled-in tensor before the kernels cost a launch of 2 us.
template <int BM>
__device__ __forceinline__ void delta_tail_zero(const AttnBwdParams &p, int b, int h, int sq, int tile) {
  const int row = tile * BM + (int)threadIdx.x;
  if (p.delta_tail && (int)threadIdx.x < BM && row >= sq && row < p.max_sq) p.delta[((int64_t)b * p.hq + h) * p.max_sq + row] = 0.f;
}

// ---- delta = rowsum(dO * O) ---------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
attn_delta_kernel(const T *__restrict__ dout, const T *__restrict__ out, float *__restrict__ delta,
                  const float *__restrict__ lse, float *__restrict__ ld2, int64_t ld2_plane, int ld2_pitch,
                  const int32_t *__restrict__ cu_q, int q_shift, int lse_pitch, int max_sq, int hq, int d, int lanes_per,
                  int64_t do_stride, int64_t o_stride, int tail) {
  constexpr int N = Vec<T>::N;
  const int b = blockIdx.y;
  const int q0 = cu_q[b] >> q_shift, sq = (cu_q[b + 1] >> q_shift) - q0;
  const int per_block = 256 / lanes_per;
  const int sub = threadIdx.x / lanes_per, ln = threadIdx.x % lanes_per;
  const int nvec = d / N;
  const int rows_ld2 = ld2 ? ((sq + 31) / 32) * 32 : sq;   // the side-by-side planes are written in whole 32-row tiles
  const int rows = tail && max_sq > rows_ld2 ? max_sq : rows_ld2;
  for (int64_t item = (int64_t)blockIdx.x * per_block + sub; item < (int64_t)rows * hq;
       item += (int64_t)gridDim.x * per_block) {
    const int i = (int)(item / hq), h = (int)(item % hq);
    if (i >= sq) {           // padding rows of the last tile: zeros, so that masked scores stay finite
      if (ln == 0 && i < rows_ld2) {
        const int64_t a2 = ((int64_t)b * hq + h) * ld2_pitch + i;
        ld2[a2] = 0.f;
        ld2[ld2_plane + a2] = 0.f;
      }
      if (tail && ln == 0 && i < max_sq) delta[((int64_t)b * hq + h) * max_sq + i] = 0.f;
      continue;
    }
    float s = 0.f;
    for (int c = ln; c < nvec; c += lanes_per) {
      const Vec<T> a = ldg(dout + (int64_t)(q0 + i) * do_stride + (int64_t)h * d + c * N);
      const Vec<T> o = ldg(out + (int64_t)(q0 + i) * o_stride + (int64_t)h * d + c * N);
#pragma unroll
      for (int j = 0; j < N; ++j) s += to_f(a.v[j]) * to_f(o.v[j]);
    }
    for (int o = lanes_per >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (ln == 0) {
      const int64_t at = ((int64_t)b * hq + h) * max_sq + i;
      delta[at] = s;
      if (ld2) {             // the copy the dK/dV kernels stream: lse in exp2 units next to delta
        const int64_t a2 = ((int64_t)b * hq + h) * ld2_pitch + i;
        ld2[a2] = lse[((int64_t)b * hq + h) * lse_pitch + i] * 1.4426950408889634f;
        ld2[ld2_plane + a2] = -s;
      }
    }
  }
}

// Sum of the head-split partials, in split order: part fp32 [hsplit][total_k][hk][d] -> dst (T, strided rows).
template <typename T>
__global__ void __launch_bounds__(256)
attn_bwd_gqa_sum_kernel(const float *__restrict__ dk_part, const float *__restrict__ dv_part, T *__restrict__ dk,
                        T *__restrict__ dv, int64_t total_k, int hk, int d, int hsplit, int64_t dk_stride,
                        int64_t dv_stride) {
  const int dv4 = d / 4;
  const int64_t nitems = total_k * hk * dv4;
  for (int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x; it < nitems; it += (int64_t)gridDim.x * 256) {
    const int cc = (int)(it % dv4);
    const int64_t r = it / dv4;
    const int h = (int)(r % hk);
    const int64_t j = r / hk;
    float4 a = make_float4(0, 0, 0, 0), bb = make_float4(0, 0, 0, 0);
    for (int s = 0; s < hsplit; ++s) {
      const int64_t off = (((int64_t)s * total_k + j) * hk + h) * d + cc * 4;
      const float4 x = *reinterpret_cast<const float4 *>(dk_part + off);
      const float4 y = *reinterpret_cast<const float4 *>(dv_part + off);
      a.x += x.x; a.y += x.y; a.z += x.z; a.w += x.w;
      bb.x += y.x; bb.y += y.y; bb.z += y.z; bb.w += y.w;
    }
    T *pk = dk + j * dk_stride + (int64_t)h * d + cc * 4;
    T *pv = dv + j * dv_stride + (int64_t)h * d + cc * 4;
    pk[0] = from_f<T>(a.x); pk[1] = from_f<T>(a.y); pk[2] = from_f<T>(a.z); pk[3] = from_f<T>(a.w);
    pv[0] = from_f<T>(bb.x); pv[1] = from_f<T>(bb.y); pv[2] = from_f<T>(bb.z); pv[3] = from_f<T>(bb.w);
  }
}

// ---------------------------------------------------------------------------------------------
// Head dim 128: direct global->LDS copies into swizzled tiles
// (no staging registers, no bank conflicts), two pipeline stages held in separate LDS
// objects, causal work made uniform by pairing tile i with tile n-1-i.
// ---------------------------------------------------------------------------------------------

}  // namespace dh

#include "attn_bwd_dkv128.h"
#include "attn_bwd_dq128.h"

namespace dh {

// dQ: 8 wavefronts = RG query row groups x SPLIT key splits (as the forward kernel); the
// partial dQ of the splits are added through LDS in split order.  As in the forward kernel
// the main loop is one rolled body whose global->LDS copies and LDS reads are written in
// assembly (scalar copy bases, XOR-derived fragment addresses, no compiler waits between
// copies in flight and reads); the copies are spread between the MFMAs.
template <typename T, int RG, int SPLIT, int BN>
__global__ void __launch_bounds__(512) attn_bwd_dq_d128_kernel(const AttnBwdParams p) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  static_assert(BN == 32, "32-key tiles");
  constexpr int D = 128, BM = 32 * RG, NS = BN / 16;
  static_assert(RG * SPLIT == 8, "8 wavefronts per workgroup");
  constexpr int TILE = BN * D;
  constexpr int SLOT = SPLIT * TILE;              // elements of one K (or V) slot: the tiles of all splits
  constexpr int SLOTB = SLOT * (int)sizeof(T);
  constexpr int BPT = BN / 4;                     // 1 KB copy blocks per tile
  constexpr int CPW = SPLIT * 2 * BPT / 8;        // copy blocks per wavefront and iteration (4 or 8)
  static_assert(CPW == 4 || CPW == 8, "copy blocks per wavefront");
  __shared__ __attribute__((aligned(1024))) T sAll[4 * SLOT];   // K slots 0..1, V slots 0..1
  __shared__ float sDel[RG * 32];                               // delta of the workgroup's rows

  const int b = seq_by_length(p.cu_q, gridDim.y, blockIdx.y);
  // the query heads of one kv head read the same K / V rows: keep a kv head on one XCD's L2
  const int ratio = p.hq / p.hk, P = gridDim.x / p.hq;
  int hkv, item;
  xcd_group_item(blockIdx.x, p.hk, ratio * P, hkv, item);
  const int h = hkv * ratio + item / P, px = item % P;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nqt = (sq + BM - 1) / BM;
  const int causal = p.causal;
  const int k_stride = (int)p.k_stride, v_stride = (int)p.v_stride;
  const float scale_log2 = p.scale_log2;
  int qt[2], nq;
  const int tiles = (p.max_sq + BM - 1) / BM;
  delta_tail_zero<BM>(p, b, h, sq, px);
  if (causal) {
    if (tiles - 1 - px != px) delta_tail_zero<BM>(p, b, h, sq, tiles - 1 - px);
    const int pair = px;
    if (2 * pair >= nqt) return;
    qt[0] = nqt - 1 - pair; qt[1] = pair;
    nq = (qt[0] == qt[1]) ? 1 : 2;
  } else {
    if (px >= nqt) return;
    qt[0] = px; qt[1] = 0; nq = 1;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: copy bookkeeping stays scalar
  const int c = lane & 31, hh = lane >> 5;
  const int rg = w % RG, sp = w / RG;
  const T *kg = reinterpret_cast<const T *>(p.k) + (int64_t)k0 * p.k_stride + (int64_t)hkv * D;
  const T *vg = reinterpret_cast<const T *>(p.v) + (int64_t)k0 * p.v_stride + (int64_t)hkv * D;
  const uint32_t ldsK = (uint32_t)(uintptr_t)sAll, ldsV = ldsK + 2 * SLOTB;

  // ---- copies: the CPW blocks of a wavefront are consecutive rows of ONE tile (K or V) -------------
  CopyLane cl0;
  cl0.l16 = lane & 15;
  cl0.lrow = lane >> 4;
  const int cp_tile = (w * CPW) / (2 * BPT);
  const int cp_v = ((w * CPW) % (2 * BPT)) / BPT;
  const int cp_r0 = 4 * ((w * CPW) % BPT);
  const int cp_stride = cp_v ? v_stride : k_stride;
  const T *cp_gt = cp_v ? vg : kg;
  const char *cp_g = reinterpret_cast<const char *>(cp_gt);
  const int cp_dst0 = cp_tile * TILE + cp_r0 * D;
  const uint32_t cp_step = (uint32_t)(4 * cp_stride) * (uint32_t)sizeof(T);
  uint32_t cp_off[4];                                 // both tiles use swz(row): chunk ^= 4 * (row % 4) + (row / 4) % 4
  {
    const uint32_t rowb = (uint32_t)(cl0.lrow * cp_stride) * (uint32_t)sizeof(T);
    const uint32_t chunk = (uint32_t)(cl0.l16 ^ (4 * cl0.lrow)) << 4;
#pragma unroll
    for (int x = 0; x < 4; ++x) cp_off[x] = rowb + (chunk ^ (uint32_t)(x << 4));
  }
  // ---- fragment reads: lane byte offsets inside a slot; other fragments by XOR / immediate offset ----
  const int r = lane & 15;
  const uint32_t rf_lane = (uint32_t)(sp * TILE * (int)sizeof(T) + c * 256 + ((hh ^ swz(c)) << 4));   // row c, chunk hh
  const int ta_x = 4 * (r >> 2) + hh;                 // transpose read of K: swz of rows 4*hh + r/4 (+8)
  const int t_lc = 2 * ((lane >> 4) & 1) + ((r & 3) >> 1);
  const uint32_t t_row = (uint32_t)(sp * TILE * (int)sizeof(T) + (4 * hh + (r >> 2)) * 256 + ((r & 3) & 1) * 8);
  const uint32_t ta_lane = t_row + (uint32_t)((t_lc ^ ta_x) << 4);
  const uint32_t tb_lane = t_row + 8 * 256 + (uint32_t)((t_lc ^ (ta_x + 2)) << 4);

  for (int qi = 0; qi < nq; ++qi) {
    const int m0 = qt[qi] * BM;
    const int wrow0 = m0 + rg * 32;
    const int row_q = wrow0 + c;
    const bool row_ok = row_q < sq;
    const int row_ld = row_ok ? row_q : sq - 1;
    Frag Qf[D / 16], dOf[D / 16];
    {
      const T *qp = reinterpret_cast<const T *>(p.q) + (int64_t)(q0 + row_ld) * p.q_stride + (int64_t)h * D;
      const T *dp = reinterpret_cast<const T *>(p.dout) + (int64_t)(q0 + row_ld) * p.do_stride + (int64_t)h * D;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        Qf[ks] = frag_ld<T>(qp + ks * 16 + 8 * hh);
        dOf[ks] = frag_ld<T>(dp + ks * 16 + 8 * hh);
      }
    }
    const float lse_c = row_ok ? p.lse[((int64_t)b * p.hq + h) * p.lse_pitch + row_q] * 1.4426950408889634f : INFINITY;
    // delta = rowsum(dO * O) of this lane's row, formed by the first key split of each row group: the lane holds
    // one half of the row's dO (its k-step chunks), reads the same chunks of O, and the two halves meet through
    // the partner lane.  The other splits get it through LDS after the barrier that publishes the first tiles.
    // Split 0 also writes it out, together with the copy the dK/dV kernel streams (lse in exp2 units next to
    // delta, zeros in the rows that pad the last 32-row tile), so that no separate pass over dO and O is
    // needed.  The dK/dV kernel therefore runs after this one.
    float del_c = 0.f;
    if (sp == 0) {
      const T *op = reinterpret_cast<const T *>(p.out) + (int64_t)(q0 + row_ld) * p.o_stride + (int64_t)h * D;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        const Frag of = frag_ld<T>(op + ks * 16 + 8 * hh);
#pragma unroll
        for (int j = 0; j < 8; ++j) del_c += to_f(dOf[ks][j]) * to_f(of[j]);
      }
      del_c += __shfl_xor(del_c, 32, 64);
      if (!row_ok) del_c = 0.f;
      if (hh == 0) {
        sDel[rg * 32 + c] = del_c;
        if (row_ok) p.delta[((int64_t)b * p.hq + h) * p.max_sq + row_q] = del_c;
        if (row_q < p.ld2_pitch) {
          const int64_t a2 = ((int64_t)b * p.hq + h) * p.ld2_pitch + row_q;
          p.ld2[a2] = row_ok ? lse_c : 0.f;
          p.ld2[p.ld2_plane + a2] = -del_c;
        }
      }
    }
    int nk_end = sk;
    if (causal && m0 + BM < nk_end) nk_end = m0 + BM;
    const int ntiles = (nk_end + BN - 1) / BN;
    const int niter = (ntiles + SPLIT - 1) / SPLIT;
    const int n_fast = sk / (SPLIT * BN);          // iterations whose tiles lie wholly inside the keys

    floatx16 dQt[D / 32];
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) dQt[t][v] = 0.f;

    if (niter > 0 && cp_tile < ntiles)
      dma_tile32_general<T, CPW>(sAll + (cp_v ? 2 * SLOT : 0) + cp_dst0, cp_gt, cp_stride, 1, cp_tile * BN + cp_r0, cp_r0, sk, cl0);
    dma_wait_all();
    __syncthreads();
    del_c = sDel[rg * 32 + c];

    const char *cp_src = nullptr;
    uint32_t cp_dst = 0;
    bool fcopy = false;
#define DH_DQ_COPY(i)                                                                                   \
    do {                                                                                                \
      if ((i) < CPW && fcopy) {                                                                         \
        __builtin_amdgcn_sched_barrier(0);                                                              \
        dma_block_fast(cp_src, cp_off[(i) & 3], cp_dst);                                                \
        cp_src += cp_step;                                                                              \
        cp_dst += 1024;                                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                              \
      }                                                                                                 \
    } while (0)

#pragma unroll 1
    for (int it = 0; it < niter; ++it) {
      const int nit = it + 1;
      const uint32_t cur = (uint32_t)((it & 1) * SLOTB), nxt = (uint32_t)((nit & 1) * SLOTB);
      const bool copy = nit < niter && nit * SPLIT + cp_tile < ntiles;
      fcopy = copy && nit < n_fast;
      cp_src = cp_g + (int64_t)((nit * SPLIT + cp_tile) * BN + cp_r0) * cp_stride * (int)sizeof(T);
      cp_dst = (cp_v ? ldsV : ldsK) + nxt + (uint32_t)(cp_dst0 * (int)sizeof(T));
      if (copy && !fcopy)
        dma_tile32_general<T, CPW>(sAll + (cp_v ? 2 * SLOT : 0) + (nit & 1) * SLOT + cp_dst0, cp_gt, cp_stride, 1,
                                   (nit * SPLIT + cp_tile) * BN + cp_r0, cp_r0, sk, cl0);
      const int tile_g = it * SPLIT + sp;
      const int n0 = tile_g * BN;
      const bool act = tile_g < ntiles && !(causal && n0 > wrow0 + 31);
      if (act) {
        uint32_t kb = ldsK + cur + rf_lane, vb = ldsV + cur + rf_lane;
        uint32_t ta = ldsK + cur + ta_lane, tb = ldsK + cur + tb_lane;
        asm volatile("" : "+v"(kb), "+v"(vb), "+v"(ta), "+v"(tb));   // derive the other addresses here, not ahead of the loop
        floatx16 S, dP;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          S[v] = 0.f;
          dP[v] = 0.f;
        }
        {
          // K and V row fragments are fetched one step ahead of the MFMAs that consume them.
          int4v fk[2], fv[2];
          lds_read128<0>(fk[0], kb);
          lds_read128<0>(fv[0], vb);
#pragma unroll
          for (int ks = 0; ks < D / 16; ++ks) {
            const int a = ks & 1, nx = (ks + 1) & 1;
            if (ks + 1 < D / 16) {
              lds_read128<0>(fk[nx], kb ^ (uint32_t)((ks + 1) << 5));
              lds_read128<0>(fv[nx], vb ^ (uint32_t)((ks + 1) << 5));
              lds_wait<2>(fk[a], fv[a]);
            } else {
              lds_wait<0>(fk[a], fv[a]);
            }
            S = M::mma(__builtin_bit_cast(Frag, fk[a]), Qf[ks], S);
            dP = M::mma(__builtin_bit_cast(Frag, fv[a]), dOf[ks], dP);
            if (CPW == 8) DH_DQ_COPY(ks);                            // all copy blocks go out in this phase, so
            if (CPW == 4 && (ks & 1)) DH_DQ_COPY(ks >> 1);           // that they have the rest of the iteration to land
          }
        }
        // dQ^T += K^T dS^T needs K^T fragments (transpose reads of the K tile): those of the first 16-key
        // step are requested now and land during the softmax part, those of the next step while the
        // current one multiplies.
        uint32_t ad[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          ad[2 * t] = ta ^ (uint32_t)(t << 6);
          ad[2 * t + 1] = tb ^ (uint32_t)(t << 6);
        }
        short4v f[2][8];
        lds_read_tr8<0>(f[0], ad);
        if ((causal && n0 + BN - 1 > wrow0) || (n0 + BN > sk)) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int kv = n0 + acc_row(v, hh);
            if (kv >= sk || (causal && kv > row_q)) S[v] = -INFINITY;     // P = dS = 0
          }
        }
        Frag dSb[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          float dsv[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int v = 8 * s + j;
            const float pe = fast_exp2(S[v] * scale_log2 - lse_c);
            dsv[j] = pe * (dP[v] - del_c);
          }
          dSb[s] = frag_pack<T>(dsv);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          short4v(&g)[8] = f[s & 1];
          if (s + 1 < NS) {
            lds_read_tr8<16 * 256>(f[(s + 1) & 1], ad);
            lds_wait<12>(g[0], g[1], g[2], g[3]);
          } else {
            lds_wait<4>(g[0], g[1], g[2], g[3]);
          }
          dQt[0] = M::mma(frag_join<T>(g[0], g[1]), dSb[s], dQt[0]);
          dQt[1] = M::mma(frag_join<T>(g[2], g[3]), dSb[s], dQt[1]);
          if (s + 1 < NS) lds_wait<8>(g[4], g[5], g[6], g[7]);
          else lds_wait<0>(g[4], g[5], g[6], g[7]);
          dQt[2] = M::mma(frag_join<T>(g[4], g[5]), dSb[s], dQt[2]);
          dQt[3] = M::mma(frag_join<T>(g[6], g[7]), dSb[s], dQt[3]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < CPW; ++i) DH_DQ_COPY(i);
      }
      dma_wait_all();
      __syncthreads();   // the next slots have landed, and everyone is done with the current ones
    }
#undef DH_DQ_COPY

    // add the splits' partial dQ through LDS, in split order: slot x = (s-1)*RG + g, 16 KB each
    float *xo = reinterpret_cast<float *>(sAll);
    static_assert((SPLIT - 1) * RG <= 6, "exchange slots");
    static_assert(4 * SLOT * sizeof(T) >= (size_t)(SPLIT - 1) * RG * 4096 * sizeof(float), "exchange area");
    if (sp > 0) {
      float *dst = xo + ((sp - 1) * RG + rg) * 4096;
#pragma unroll
      for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[(t * 16 + v) * 64 + lane] = dQt[t][v];
    }
    __syncthreads();
    if (sp == 0) {
#pragma unroll
      for (int s2 = 1; s2 < SPLIT; ++s2) {
        const float *src = xo + ((s2 - 1) * RG + rg) * 4096;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) dQt[t][v] += src[(t * 16 + v) * 64 + lane];
      }
      if (row_ok) {
        T *dqp = reinterpret_cast<T *>(p.dq) + (int64_t)(q0 + row_q) * p.dq_stride + (int64_t)h * D;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
          for (int vb = 0; vb < 4; ++vb) {
            struct alignas(8) { T v[4]; } a;
            if (p.dq_accumulate) {
              a = *reinterpret_cast<const decltype(a) *>(dqp + 32 * t + 8 * vb + 4 * hh);
#pragma unroll
              for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(static_cast<float>(a.v[e]) + dQt[t][4 * vb + e] * p.scale);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(dQt[t][4 * vb + e] * p.scale);
            }
            *reinterpret_cast<decltype(a) *>(dqp + 32 * t + 8 * vb + 4 * hh) = a;
          }
      }
    }
    __syncthreads();
  }
}

// dQ from the dS blocks that the dK/dV kernel left in the workspace: dQ^T[d, q] += K^T[d, key] dS^T[key, q], one
// matrix product instead of the three of the recomputing kernel above (which stays for shapes whose dS would not
// fit the workspace).  Same workgroup shape: 2 query row groups x 4 key splits, 32-key steps, the splits' partial
// sums added through LDS in split order.  A step needs the K tile of its split (8 KB, swizzled rows, transpose
// reads as above) and one 2 KB dS block per row group, copied as it lies in memory; its transpose reads pick,
// for a 16-lane group of query columns, the 8-byte pieces (u, hh) of four consecutive keys, which puts query
// row n of the tile on lane n.  The kernel streams 2 bytes of dS per 256 flops: it is bound by memory.
template <typename T>
__global__ void __launch_bounds__(512) attn_bwd_dq2_d128_kernel(const AttnBwdParams p) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  constexpr int D = 128, RG = 2, SPLIT = 4, BN = 32, BM = 32 * RG;
  constexpr int TILE = BN * D;                         // elements of one K tile
  constexpr int TILEB = TILE * (int)sizeof(T);
  constexpr int SLOTB = SPLIT * TILEB;                 // the K tiles of all splits: one stage
  constexpr int DSB = RG * 2048;                       // the dS blocks of one split (one per row group)
  constexpr int DSLOTB = SPLIT * DSB;
  constexpr int NST = 3;                               // stages: the copies of a step go out two steps ahead of it
  __shared__ __attribute__((aligned(1024))) char sAll[NST * SLOTB + NST * DSLOTB];   // 144 KB

  const int b = seq_by_length(p.cu_q, gridDim.y, blockIdx.y);
  // a head's dS blocks were written from one XCD (the dK/dV kernel keeps a head group there): read them from the
  // same one; the K rows of the kv head are small next to them
  const int ratio = p.hq / p.hk, P = gridDim.x / p.hq;
  int h, px;
  xcd_group_item(blockIdx.x, p.hq, P, h, px);
  const int hkv = h / ratio;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nqt = (sq + BM - 1) / BM;
  const int causal = p.causal;
  const int k_stride = (int)p.k_stride;
  int qt[2], nq;
  if (causal) {
    if (2 * px >= nqt) return;
    qt[0] = nqt - 1 - px; qt[1] = px;
    nq = (qt[0] == qt[1]) ? 1 : 2;
  } else {
    if (px >= nqt) return;
    qt[0] = px; qt[1] = 0; nq = 1;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int rg = w % RG, sp = w / RG;
  const T *kg = reinterpret_cast<const T *>(p.k) + (int64_t)k0 * p.k_stride + (int64_t)hkv * D;
  const char *kg_b = reinterpret_cast<const char *>(kg);
  const uint32_t ldsK = (uint32_t)(uintptr_t)sAll, ldsD = ldsK + NST * SLOTB;

  // ---- copies of wavefront w: rows [16 half, 16 half + 16) of the K tile of split w / 2 (four 1 KB blocks) and the
  // dS block of row group `half` of that split (two 1 KB blocks) -------------------------------------------------
  CopyLane cl0;
  cl0.l16 = lane & 15;
  cl0.lrow = lane >> 4;
  const int csp = w >> 1, half = w & 1;
  const uint32_t cp_step = (uint32_t)(4 * k_stride) * (uint32_t)sizeof(T);
  uint32_t cp_off[4];
  {
    const uint32_t rowb = (uint32_t)(cl0.lrow * k_stride) * (uint32_t)sizeof(T);
    const uint32_t chunk = (uint32_t)(cl0.l16 ^ (4 * cl0.lrow)) << 4;
#pragma unroll
    for (int x = 0; x < 4; ++x) cp_off[x] = rowb + (chunk ^ (uint32_t)(x << 4));
  }
  // The dK/dV kernel wrote a dS block as two fragments of 64 lanes x 16 bytes (piece 64 s + L is lane L of fragment
  // s).  The transpose reads below fetch, per instruction, the pieces L = 32 b + 8 t + 4 hh + j of both fragments
  // (t fixed; j = 0..3, b = 0..1): copied as they lie, the four 64-byte runs (s, b) of a half wavefront fall on the
  // same 16 banks.  So the copy permutes: LDS position 64 hh + 16 t + 8 s + 4 b + j holds that piece (lane l of the
  // copy for half hh fetches the piece with j = l % 4, b = l / 4 % 2, s = l / 8 % 2, t = l / 16), and the 16 pieces of
  // a half wavefront's read are 256 consecutive bytes.
  const uint32_t ds_lane = 16u * (uint32_t)(64 * ((lane >> 3) & 1) + 32 * ((lane >> 2) & 1) + 8 * ((lane >> 4) & 3) + (lane & 3));
  const int64_t ds_head = ((int64_t)b * p.hq + h) * p.ds_nqt;
  const char *ds_b = reinterpret_cast<const char *>(p.ds);

  // ---- fragment reads ------------------------------------------------------------------------------------------
  const int r = lane & 15;
  const int ta_x = 4 * (r >> 2) + hh;                 // transpose reads of K: swz of rows 4*hh + r/4 (+8)
  const int t_lc = 2 * ((lane >> 4) & 1) + ((r & 3) >> 1);
  const uint32_t t_row = (uint32_t)(sp * TILEB + (4 * hh + (r >> 2)) * 256 + ((r & 3) & 1) * 8);
  const uint32_t ta_lane = t_row + (uint32_t)((t_lc ^ ta_x) << 4);
  const uint32_t tb_lane = t_row + 8 * 256 + (uint32_t)((t_lc ^ (ta_x + 2)) << 4);
  // dS block: piece (s = 16-lane group, hh_p = r % 2) of key 4 hh + r / 4, half u = (r % 4) / 2 of the piece
  const uint32_t db_lane = (uint32_t)(sp * DSB + rg * 2048 + ((64 * hh + 8 * ((lane >> 4) & 1) + 4 * (r & 1) + (r >> 2)) * 16) +
                                      ((r & 3) >> 1) * 8);        // + 256 t

  for (int qi = 0; qi < nq; ++qi) {
    const int m0 = qt[qi] * BM;
    const int wrow0 = m0 + rg * 32;
    const int row_q = wrow0 + c;
    const bool row_ok = row_q < sq;
    int nk_end = sk;
    if (causal && m0 + BM < nk_end) nk_end = m0 + BM;
    const int ntiles = (nk_end + BN - 1) / BN;
    const int niter = (ntiles + SPLIT - 1) / SPLIT;
    const int n_fast = sk / (SPLIT * BN);          // iterations whose K tiles lie wholly inside the keys
    const int64_t ds_row = (ds_head + (m0 >> 5) + half) * p.ds_nkb;   // the copied block row: query tile of row group `half`

    floatx16 dQt[D / 32];
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) dQt[t][v] = 0.f;

    auto issue = [&](int it) {
      const int tile = it * SPLIT + csp;
      if (tile >= ntiles) return;
      const uint32_t stK = (uint32_t)((it % NST) * SLOTB), stD = (uint32_t)((it % NST) * DSLOTB);
      if (it < n_fast) {
        const char *src = kg_b + (int64_t)(tile * BN + 16 * half) * k_stride * (int)sizeof(T);
        uint32_t dst = ldsK + stK + (uint32_t)(csp * TILEB + 16 * half * 256);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          dma_block_fast(src, cp_off[x], dst);
          src += cp_step;
          dst += 1024;
        }
      } else {
        dma_tile32_general<T, 4>(reinterpret_cast<T *>(sAll + stK + csp * TILEB) + 16 * half * D, kg, k_stride, 1,
                                 tile * BN + 16 * half, 16 * half, sk, cl0);
      }
      const char *dsrc = ds_b + (ds_row + tile) * 2048;
      const uint32_t ddst = ldsD + stD + (uint32_t)(csp * DSB + half * 2048);
      dma_block_fast(dsrc, ds_lane, ddst);
      dma_block_fast(dsrc + 64, ds_lane, ddst + 1024);
    };

    // Steps 0 and 1 go out now; in the loop, step it + 2 goes out at the top of step it and the wait at the bottom
    // leaves the newest step's copies in flight (6 per wavefront, or none: vmcnt counts in issue order).
    if (niter > 0) issue(0);
    if (niter > 1) issue(1);
    if (niter > 1 && 1 * SPLIT + csp < ntiles && 1 < n_fast) {
      asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      dma_wait_all();
      __syncthreads();
    }

#pragma unroll 1
    for (int it = 0; it < niter; ++it) {
      if (it + 2 < niter) issue(it + 2);              // has two steps to land
      const int tile_g = it * SPLIT + sp;
      const int n0 = tile_g * BN;
      const bool act = tile_g < ntiles && !(causal && n0 > wrow0 + 31);
      if (act) {
        const uint32_t curK = ldsK + (uint32_t)((it % NST) * SLOTB), curD = ldsD + (uint32_t)((it % NST) * DSLOTB);
        uint32_t ta = curK + ta_lane, tb = curK + tb_lane, db = curD + db_lane;
        asm volatile("" : "+v"(ta), "+v"(tb), "+v"(db));
        // LDS reads in assembly (the compiler would hold them behind every copy in flight): the four dS pieces,
        // the K^T fragments of the first 16 keys, then those of the second while the first multiply
        uint32_t ad[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          ad[2 * t] = ta ^ (uint32_t)(t << 6);
          ad[2 * t + 1] = tb ^ (uint32_t)(t << 6);
        }
        short4v bq[4], f0[8], f1[8];
        lds_read_tr4<256>(bq, db);
        lds_read_tr8<0>(f0, ad);
        lds_wait<4>(bq[0], bq[1], bq[2], bq[3]);
        lds_wait<4>(f0[0], f0[1], f0[2], f0[3]);
        lds_read_tr8<16 * 256>(f1, ad);
        const Frag dS0 = frag_join<T>(bq[0], bq[1]), dS1 = frag_join<T>(bq[2], bq[3]);
        dQt[0] = M::mma(frag_join<T>(f0[0], f0[1]), dS0, dQt[0]);
        dQt[1] = M::mma(frag_join<T>(f0[2], f0[3]), dS0, dQt[1]);
        lds_wait<8>(f0[4], f0[5], f0[6], f0[7]);
        dQt[2] = M::mma(frag_join<T>(f0[4], f0[5]), dS0, dQt[2]);
        dQt[3] = M::mma(frag_join<T>(f0[6], f0[7]), dS0, dQt[3]);
        lds_wait<4>(f1[0], f1[1], f1[2], f1[3]);
        dQt[0] = M::mma(frag_join<T>(f1[0], f1[1]), dS1, dQt[0]);
        dQt[1] = M::mma(frag_join<T>(f1[2], f1[3]), dS1, dQt[1]);
        lds_wait<0>(f1[4], f1[5], f1[6], f1[7]);
        dQt[2] = M::mma(frag_join<T>(f1[4], f1[5]), dS1, dQt[2]);
        dQt[3] = M::mma(frag_join<T>(f1[6], f1[7]), dS1, dQt[3]);
      }
      // step it + 1 must have landed; the copies of step it + 2 (the newest 6 of this wavefront, if it issued them
      // in the fast form) may stay in flight
      // (__syncthreads() would drain them: it waits for every memory operation before its barrier)
      if (it + 2 < niter && (it + 2) * SPLIT + csp < ntiles && it + 2 < n_fast) {
        asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      } else {
        dma_wait_all();
        __syncthreads();
      }
    }

    // add the splits' partial dQ through LDS, in split order: slot x = (s-1)*RG + g, 16 KB each
    float *xo = reinterpret_cast<float *>(sAll);
    static_assert(sizeof(sAll) >= (size_t)(SPLIT - 1) * RG * 4096 * sizeof(float), "exchange area");
    if (sp > 0) {
      float *dst = xo + ((sp - 1) * RG + rg) * 4096;
#pragma unroll
      for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[(t * 16 + v) * 64 + lane] = dQt[t][v];
    }
    __syncthreads();
    if (sp == 0) {
#pragma unroll
      for (int s2 = 1; s2 < SPLIT; ++s2) {
        const float *src = xo + ((s2 - 1) * RG + rg) * 4096;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) dQt[t][v] += src[(t * 16 + v) * 64 + lane];
      }
      if (row_ok) {
        T *dqp = reinterpret_cast<T *>(p.dq) + (int64_t)(q0 + row_q) * p.dq_stride + (int64_t)h * D;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
          for (int vb = 0; vb < 4; ++vb) {
            struct alignas(8) { T v[4]; } a;
            if (p.dq_accumulate) {
              a = *reinterpret_cast<const decltype(a) *>(dqp + 32 * t + 8 * vb + 4 * hh);
#pragma unroll
              for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(static_cast<float>(a.v[e]) + dQt[t][4 * vb + e] * p.scale);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) a.v[e] = static_cast<T>(dQt[t][4 * vb + e] * p.scale);
            }
            *reinterpret_cast<decltype(a) *>(dqp + 32 * t + 8 * vb + 4 * hh) = a;
          }
      }
    }
    __syncthreads();
  }
}

template <typename T>
static int launch_dq2_d128(const AttnBwdParams &p, int batch, hipStream_t st) {
  constexpr int BM = 64;
  const int nqt = (int)cdiv(p.max_sq, BM);
  dim3 grid((unsigned)((p.causal ? (nqt + 1) / 2 : nqt) * p.hq), (unsigned)batch);
  hipLaunchKernelGGL((attn_bwd_dq2_d128_kernel<T>), grid, dim3(512), 0, st, p);
  return DH_OK;
}

template <typename T, int RG>
static int launch_dq128(const AttnBwdParams &p, int batch, hipStream_t st) {
  const int nqt = (int)cdiv(p.max_sq, 64 * RG);
  dim3 grid((unsigned)((p.causal ? (nqt + 1) / 2 : nqt) * p.hq), (unsigned)batch);
  hipLaunchKernelGGL((attn_bwd_dq128_kernel<T, RG>), grid, dim3(256), 0, st, p);
  return DH_OK;
}

template <typename T, int RG, int SPLIT, int BN>
static int launch_dq_d128(const AttnBwdParams &p, int batch, hipStream_t st) {
  constexpr int BM = 32 * RG;
  const int nqt = (int)cdiv(p.max_sq, BM);
  dim3 grid((unsigned)((p.causal ? (nqt + 1) / 2 : nqt) * p.hq), (unsigned)batch);
  hipLaunchKernelGGL((attn_bwd_dq_d128_kernel<T, RG, SPLIT, BN>), grid, dim3(512), 0, st, p);
  return DH_OK;
}

template <typename T>
static int launch_dkv_d128(const AttnBwdParams &p, int batch, int max_sk, hipStream_t st) {
  const int nkt = (int)cdiv(max_sk, 64);
  dim3 grid((unsigned)((p.causal ? (nkt + 1) / 2 : nkt) * p.hk * p.hsplit), (unsigned)batch);
  if (p.ds) hipLaunchKernelGGL((attn_bwd_dkv128_kernel<T, true>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((attn_bwd_dkv128_kernel<T, false>), grid, dim3(256), 0, st, p);
  return DH_OK;
}

}  // namespace dh

#include "attn_bwd_tile.h"

namespace dh {

// ---- host -------------------------------------------------------------------------------------
// Query heads of a kv head are split over workgroups (each with fp32 partial dK / dV that a second kernel adds up)
// only as far as it takes to give every compute unit one workgroup: beyond that the partials cost more than the
// finer grain gives (ring step, 32 q / 8 kv heads: 4 splits 669 us, 2 splits 633 us, none 609 us).
static int pick_hsplit(int64_t blocks, int hq, int hk) {
  const int ratio = hq / hk;
  int hsplit = 1;
  for (int s = 1; s <= ratio; ++s)
    if (ratio % s == 0 && blocks * s <= 256) hsplit = s;
  return hsplit;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

template <typename T>
static int launch_delta(const void *dout, const void *out, float *delta, const float *lse, float *ld2, int64_t ld2_plane,
                        int ld2_pitch, const int32_t *cu_q, int q_shift, int lse_pitch, int batch, int max_sq, int hq, int d,
                        int64_t do_stride, int64_t o_stride,
                        int tail, hipStream_t st) {
  const int nvec = d / Vec<T>::N;
  int lanes_per = 1;
  while (lanes_per < nvec && lanes_per < 64) lanes_per <<= 1;
  const int per_block = 256 / lanes_per;
  int64_t blocks = cdiv((int64_t)(ld2 ? ld2_pitch : max_sq) * hq, per_block);
  if (blocks > 256 * 16) blocks = 256 * 16;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL((attn_delta_kernel<T>), dim3((unsigned)blocks, (unsigned)batch), dim3(256), 0, st,
                     (const T *)dout, (const T *)out, delta, lse, ld2, ld2_plane, ld2_pitch, cu_q, q_shift, lse_pitch, max_sq, hq, d, lanes_per,
                     do_stride, o_stride, tail);
  return DH_OK;
}

int attn_bwd_f32(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                 void *dq, void *dk, void *dv, const int32_t *cu_q, const int32_t *cu_k, int batch, int max_sq,
                 int max_sk, int hq, int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                 int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride, float scale, int causal,
                 int dq_accumulate, hipStream_t st);

constexpr int DKV_ROWS = 64;  // key rows of a dK/dV workgroup

// Keeping dS for the dQ product costs 2 bytes per (head, query, key) of workspace, written once and read once.
// It pays where the recomputing dQ kernel runs its small-grid form (fewer than 256 workgroups of 128 query rows: whole backward, us,
// recomputing / keeping: the 8-head shard at 4096 tokens 149 / 122, at 2048 tokens 86 / 71); with the chip full the recomputing
// kernel is the faster one (32 heads x 4096 386 / 479; 16 heads 217 / 275), as the extra memory traffic then costs more
// than the two products saved.  Above the byte limit dS is never kept.
static std::atomic<size_t> g_ds_limit{(size_t)1280 << 20};
static std::atomic<int> g_ds_when_full{0};   // 1: keep dS also where the recomputing dQ kernel would fill the chip

// Whether the recomputing dQ kernel would fill the chip (its 128-row form).
static bool dq_big_grid(int batch, int max_sq, int hq, int causal) {
  return attn_wgs(max_sq, 128, hq, batch, causal) >= ATTN_128ROW_MIN_WG;
}

// Head dim 128 with short sequences and little to do altogether: the kernels of the other head dims start and end sooner
// than the hand-ordered ones, and dS is not kept.  Backward, us, hand-ordered / other (two launches): causal, query rows times heads up to
// 16384: 32 heads x 100 32 / 22, 8 x 300 36 / 28, 32 x 500 44 / 37, 8 x 8 x 256 40 / 29; above: 64 heads x 300 41 / 47, 16 x 4 x
// 300 42 / 48, 32 x 32 x 300 456 / 491, 20 to 470 tokens x 32 heads 81 / 86.  Not causal only the shortest: 12 heads x 19
// 18.5 / 16.2, 4 x 34 19.1 / 17.2, but 8 x 169 + 18 23 / 25, 16 x 22 to 326 30 / 32.  (512 rows and more: 56 / 76 at 32 x 2 x 512.)
static bool bwd_short(int max_sq, int max_sk, int causal, int64_t total_q, int hq) {
  if (max_sq >= 512 || max_sk >= 512) return false;
  return causal ? total_q * hq <= 16384 : max_sq <= 48 && max_sk <= 48;
}

// Key splits of a GQA group over workgroups.  The hand-ordered causal dK/dV kernel takes two key tiles a workgroup.
static int bwd_hsplit(int max_sk, int batch, int hq, int hk, bool paired) {
  return pick_hsplit(cdiv(paired ? (max_sk + 1) / 2 : max_sk, DKV_ROWS) * hk * batch, hq, hk);
}

// Whether dK/dV and dQ go into one launch of the tile kernels, behind the delta kernel (2 us).  Either pass alone leaves
// compute units idle: all of those that it has no workgroup for, the last round's, and with causal rows those that got short
// tiles (one workgroup a compute unit in all forms: registers).  Together the long workgroups (dK/dV: 1.3 times a dQ one and
// once per query head of its group) start first and the others fill in.  `a` and `b`: workgroups of dQ and dK/dV with work.
// Backward, us, two launches / one, head dims 64 | 192 (96 and 256 behave as they do):
//   all in one round: 16 heads x 300 17.4 / 13.3 | 40 / 26, causal or not;
//   causal, a round and a half: 8 x 1500 36.9 / 24.9 | 118 / 66, 32 x 300 17.9 / 17.0 | 42 / 35; two full rounds of short rows
//     16 x 16 x 60 15.9 / 17.8 | 29 / 32, of long ones 8 x 2048 45 / 34 | 152 / 102, 16 x 1024 29.0 / 28.2 | 88 / 83; dK/dV in one
//     round, dQ in several: 32 query / 8 kv heads x 1500 93 / 67 | 315 / 218, but 16 x 1500 (dK/dV in two) 42.7 / 44.4 | 123 / 127;
//   otherwise by the model: 16 x 1500 not causal (1.28 predicted) 71 / 58 | 234 / 183, 32 / 8 x 600 + 300 (1.38) 49 / 37 | 152 / 100, 32
//     x 300 (1.15, not taken) 18.8 / 18.5 | 42 / 42, 16 x 1024 (1.0) 29.3 / 30.9 | 89 / 93.
// Head dim 128 has the hand-ordered kernels to compare with, whose workgroups start and end later but run 1.5 times as fast:
//   one round: 16 x 300 36 / 20 causal, 26 / 20 not, 8 x 1024 48 / 36 causal, 38 / 36 not;
//   causal, up to a round and a half: 8 x 1500 58 / 48; two: 32 x 512 44 / 41, 16 x 1024 52 / 57, 16 x 16 x 60 22.9 / 22.6; not
//   causal: 8 x 1500 50 / 86, 32 x 512 35 / 42.
// A group split eight ways from 512 rows on (8 query / 1 kv head x 1024: 55 / 43) and rectangular calls of several sequences that
// are not causal stay with the hand-ordered kernels: callers size the workspace there to choose between their two forms of dQ.
// Few query rows of many keys are not for it either: dQ is a long chain of key tiles for a few workgroups here and a product over kept dS
// there: 8 query / 1 kv head x 27 rows x 5086 keys 55 / 124, 4 / 2 x 66 x 918 29 / 34, 1 / 1 x 363 x 1427 31 / 42, 1423 x 2767 50 / 71, but
// 12 / 4 x 193 x 450 32 / 27.  (The line was drawn against a dK/dV of eight wavefronts.  With the present one long rows of few heads that are not
// causal are slower here: 1 / 1 x 1500 x 2000 46 / 55, 1833 x 2547 53 / 66, 3000 x 20 50 / 77, 2 / 2 x 4000 86 / 105, but 4 / 4 x 1500 47 / 48.)
// A group that is left in pieces of several heads makes dK/dV's workgroups that much longer: from 512 rows on not here.  One
// long sequence among short ones, hand-ordered / here: 12 query / 4 kv heads x 791 + 76 + 32 54 / 41, 4 / 2 x 2746 + 7 81 / 80 (with the
// splits of the grid laid out for the longest instead of those of the work, whole calls, 57 -> 86 and 117 -> 168).
// A batch of one long sequence and many short ones has a grid for 128-row tiles, most of it empty, and the work of a few 64-row
// ones.  Backward, hand-ordered / two launches of the tile kernels / one: 8 heads, 1000 rows and 7 x 1 58 / 62 / 47, 4 query / 2 kv heads, 2163 and 7 x
// 2 109 / 157 / 73, 12 / 4, 386 + 382 and 14 x 1 50 / 59 / 45.  Of 99 such batches of up to 24 sequences 5 were slower in one launch (by up to
// 7 %); of 51 larger ones 17, by up to a third (4 heads, 599 and 47 x 1 49 / 58 / 68; 4 / 2, 451 and 31 x 3 52 / 56 / 67): not there.  At the
// other head dims, where the two launches are these kernels too, such batches keep the 128-row dQ tiles.
static bool dq_tile_fills(int max_sq, int hq, int batch) { return attn_wgs(max_sq, 128, hq, batch, 0) >= 2 * 256; }
struct BwdBoth { bool pays; int hsplit; };      // key splits of a GQA group: by the workgroups with work
static BwdBoth bwd_both(int batch, int max_sq, int max_sk, int64_t total_q, int64_t total_k, int hq, int hk, int d, int causal) {
  if (max_sq <= 0 || max_sk <= 0) return {false, 1};
  auto tiles = [&](int longest, int64_t total) {
    const int64_t grid = cdiv(longest, 64) * batch, real = total / 64 + batch;
    return grid < real ? grid : real;
  };
  int hs = pick_hsplit(tiles(max_sk, total_k) * hk, hq, hk);
  // A group of few heads and rows stays whole where that is an iteration or two more for its workgroup (each of 128 query rows,
  // 64 from head dim 128 on): the sum of the pieces is a launch of 2.5 us.  us, split / whole, causal: 4 query / 2 kv heads x 60 rows,
  // head dim 64 12.5 / 11.2, 96 14.7 / 13.3, 128 15.2 / 14.2, 256 25.0 / 26.3; 12 / 4 x 60 13.1 / 12.6, 15.2 / 15.3, 15.8 / 16.3; 16 / 4 x 60 13.4 / 13.7.
  if (hs == hq / hk && (hs - 1) * cdiv(max_sq, d < 128 ? 128 : 64) <= (d == 64 ? 2 : d <= 128 ? 1 : 0)) hs = 1;
  const int64_t a = tiles(max_sq, total_q) * hq, b = tiles(max_sk, total_k) * hk * hs;
  if (d == 128) {
    if (batch > 24 && dq_tile_fills(max_sq, hq, batch)) return {false, hs};
    if (max_sq >= 512 && (hs >= 8 || hs < hq / hk)) return {false, hs};      // (512 rows are never left whole above)
    if (!causal) return {a + b <= 256 && (max_sq == max_sk || (batch == 1 && (max_sk <= 600 || 2 * (int64_t)max_sk <= 3 * (int64_t)max_sq))), hs};
    return {a + b <= 384 || (a + b <= 512 && max_sq >= 256 && max_sq < 1024), hs};
  }
  if (a + b <= (causal ? 384 : 256)) return {true, hs};
  if (causal && max_sq >= 1024) return {b <= 256, hs};
  // rounds of 256, in units of a dQ workgroup's time: one pass after the other, and both with the dK/dV workgroups first
  const double rho = 1.3 * (hq / hk / hs), apart = (double)cdiv(a, 256) + (double)cdiv(b, 256) * rho;
  const int64_t full = b / 256, more = b % 256;
  auto room = [&](double t) {        // dQ workgroups that end by t
    const double x = t - (double)full * rho, y = x - rho;
    return (x > 0 ? (int64_t)x * (256 - more) : 0) + (y > 0 ? (int64_t)y * more : 0);
  };
  const double t = apart / 1.2;
  return {t >= (double)cdiv(b, 256) * rho && room(t) >= a, hs};
}

// Query rows of a tile of recomputing dQ where 128-row tiles fill the chip: 256 or 128 on one wavefront a SIMD, or 0: 128 on eight wavefronts.
// What ends first by this count, in thousands of cycles: a tile's rows are loaded and stored in 15 and 16.5 where the eight wavefronts take
// 9, a tile of 32 keys takes 1.9 for 256 rows or, in two splits, 0.96 for 128 (eight wavefronts 1.8); workgroups run in rounds of 256, a
// last one that is not full ends sooner, and those of several lengths fill each other's (not causal: 6 % better on one wavefront than the count
// says).  Fitted to 504 whole backward calls of random sizes that the forms tell apart: 1.0 % slower than the best of the three, none slower
// than on eight wavefronts throughout; a line at 208 workgroups of either tile was 4.3 % and 27.  us, eight wavefronts / 128 / 256 rows, not
// causal: 16 query / 4 kv heads x 12 x 140 46 / 47 / 36, 64 / 8 x 32 of up to 183 271 / 247 / 212, 32 / 8 x 5 x 908 273 / 261 / 250, 64 / 8 x 24 x 56
// 71 / 89 / 92, 32 / 32 x 16 x 56 39 / 47 / 49; causal: 32 / 32 x 12 of up to 1591 851 / 819 / 781, 64 / 8 x 8 x 631 350 / 365 / 363, 24 / 8 x 24 x 765 513 / 526 / 539.
static int dq_rows(int max_sq, int max_sk, int64_t total_q, int64_t total_k, int hq, int batch, int causal) {
  const double bound = (double)batch * max_sq, q = (double)total_q < bound ? (double)total_q : bound;
  const bool ragged = 10 * q < 9 * bound;
  auto cycles = [&](int rows, double ends, double tile) {
    const int64_t t = cdiv(max_sq, rows);
    double wgs = (double)attn_wgs(max_sq, rows, hq, batch, causal), keys = (double)max_sk / 32;
    if (ragged) wgs = std::min(wgs, (causal ? (q / rows + batch) / 2 : q / rows + 0.5 * batch) * hq);
    if (causal) {                                     // of two tiles i and n - 1 - i, or of the only one
      keys = (double)((t > 1 ? t + 1 : 1) * rows / 32 - (t * rows - max_sq) / 32);
      if (ragged) keys = std::min(keys, (1.5 * q / batch + rows) / 32);
      if (t > 1) ends *= 2;
    } else if (ragged) {
      keys = (double)total_k / batch / 32;
    }
    const double x = wgs / 256;
    return (x <= 1 ? 1 : ragged ? x + 0.05 : 0.5 * std::ceil(x) + 0.5 * x) * (ends + keys * tile);
  };
  const double one = ragged && !causal ? 0.94 : 1;
  const double w8 = cycles(128, 9.0, 1.8), w4 = one * cycles(256, 15.0, 1.86), w2 = one * cycles(128, 16.5, 0.96);
  return w8 <= w4 && w8 <= w2 ? 0 : w4 <= w2 ? 256 : 128;
}

// What one 16-bit call runs.
struct AttnBwdRoute {
  bool keep_ds;      // dK/dV keeps dS and dQ is one product over it; else dQ recomputes, first, and forms delta
  bool hand_dkv, hand_dq;      // head dim 128's hand-ordered kernels
  bool big_dq;       // 128-row query tiles in dQ
  int dq_rows;       // ... of the hand-ordered kernels: tiles of 256 or 128 rows on one wavefront a SIMD, or 0: the one of eight wavefronts
  bool both;         // dK/dV and dQ in one launch of the tile kernels, behind the delta kernel
  int hsplit;        // workgroups that share a GQA group in dK/dV
};
// `wide`: token strides that the 32-bit copy offsets of the hand-ordered kernels do not reach across a tile.
static AttnBwdRoute attn_bwd_route(int batch, int max_sq, int max_sk, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                                   int causal, bool room_for_ds, bool wide = false) {
  const BwdBoth both = bwd_both(batch, max_sq, max_sk, total_q, total_k, hq, hk, d, causal);
  const bool short_rows = d == 128 && (both.pays || wide || bwd_short(max_sq, max_sk, causal, total_q, hq)), big = dq_big_grid(batch, max_sq, hq, causal);
  AttnBwdRoute r;
  r.keep_ds = room_for_ds && max_sk > 0 && !short_rows;
  r.hand_dkv = d == 128 && !short_rows;
  r.hand_dq = r.hand_dkv && (!causal || !big || attn_causal_fills(max_sq, hq, batch, total_q));
  const bool fills = d <= 128 && dq_tile_fills(max_sq, hq, batch);
  r.both = both.pays && (d == 128 || !fills);
  r.big_dq = r.hand_dq ? big : fills && !r.both;
  r.dq_rows = r.hand_dq && big ? dq_rows(max_sq, max_sk, total_q, total_k, hq, batch, causal) : 0;
  r.hsplit = r.both ? both.hsplit : bwd_hsplit(max_sk, batch, hq, hk, d == 128 && causal);
  return r;
}

// The kernels behind delta of one call.
template <typename T, int D>
static int bwd_passes(const AttnBwdParams &p, const AttnBwdRoute &r, int batch, int max_sq, int max_sk, hipStream_t st) {
  int rc = DH_OK;
  // recomputing dQ kernels form delta and run first
  if (r.both) {
    if constexpr (D < 128) rc = launch_both_tile<T, D, 2, 4, 2, 4, 2>(p, batch, max_sk, st);
    else rc = launch_both_tile<T, D, 2, 2, 2, 2, 1>(p, batch, max_sk, st);
  } else if (max_sq > 0 && !r.keep_ds) {
    if constexpr (D == 128) {
      if (r.hand_dq) rc = r.big_dq ? (r.dq_rows == 256 ? launch_dq128<T, 4>(p, batch, st) : r.dq_rows == 128 ? launch_dq128<T, 2>(p, batch, st) : launch_dq_d128<T, 4, 2, 32>(p, batch, st)) : launch_dq_d128<T, 2, 4, 32>(p, batch, st);
      else rc = r.big_dq ? launch_dq_tile<T, D, 4, 2, 2>(p, batch, st) : launch_dq_tile<T, D, 2, 4, 2>(p, batch, st);
    } else if constexpr (D < 128) {
      rc = r.big_dq ? launch_dq_tile<T, D, 4, 2, D == 64 ? 4 : 2>(p, batch, st) : launch_dq_tile<T, D, 2, 4, 2>(p, batch, st);
    } else {
      rc = launch_dq_tile<T, D, 2, 2, 1>(p, batch, st);
    }
  }
  if (rc == DH_OK && max_sk > 0 && !r.both) {
    if constexpr (D == 128) rc = r.hand_dkv ? launch_dkv_d128<T>(p, batch, max_sk, st) : launch_dkv_tile<T, D, 2, 2, 1>(p, batch, max_sk, st);
    else if constexpr (D < 128) rc = launch_dkv_tile<T, D, 2, 4, 2>(p, batch, max_sk, st);
    else rc = launch_dkv_tile<T, D, 2, 2, 1>(p, batch, max_sk, st);
  }
  if (rc == DH_OK && p.hsplit > 1 && p.total_k > 0) {
    int64_t blocks = cdiv(p.total_k * p.hk * (D / 4), 256);
    if (blocks > 256 * 16) blocks = 256 * 16;
    hipLaunchKernelGGL((attn_bwd_gqa_sum_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, st, p.dk_part, p.dv_part, (T *)p.dk,
                       (T *)p.dv, p.total_k, p.hk, D, p.hsplit, p.dk_stride, p.dv_stride);
  }
  if constexpr (D == 128) {
    if (rc == DH_OK && max_sq > 0 && r.keep_ds) rc = launch_dq2_d128<T>(p, batch, st);
  }
  return rc;
}

// Bytes of the dS blocks for these sizes (key count as an upper bound of the longest sequence); 0 for calls that
// never keep dS, whatever space there is (other head dims, fp32, a chip-filling recomputing kernel).
static size_t ds_bytes_wanted(int batch, int max_sq, int64_t max_sk, int hq, int d, int dtype, int causal) {
  if (dtype == DH_F32 || d != 128 || batch <= 0 || max_sq <= 0 || max_sk <= 0) return 0;
  if (dq_big_grid(batch, max_sq, hq, causal) && !g_ds_when_full.load()) return 0;
  // one block more per row than needed: rows a power of two apart would meet on the same memory channels
  const size_t nqt = 2 * (size_t)cdiv(max_sq, 64), nkb = 2 * (size_t)cdiv(max_sk, 64) + 1;
  return (size_t)batch * hq * nqt * nkb * 2048;
}

// ... and under the process-wide limit: 0 if they exceed it.
static size_t ds_bytes(int batch, int max_sq, int64_t max_sk, int hq, int d, int dtype, int causal) {
  const size_t n = ds_bytes_wanted(batch, max_sq, max_sk, hq, d, dtype, causal);
  return n <= g_ds_limit.load() ? n : 0;
}

// Workspace bytes every call of these sizes needs: delta, the lse / delta planes of the head-dim-128 kernels and the
// fp32 dK / dV partials of a split GQA group.  The dS blocks, where kept, lie behind them.
static size_t bwd_base_bytes(int64_t total_k, int batch, int max_seqlen_q, int hq, int hk, int d, int dtype) {
  const size_t sq = (size_t)(max_seqlen_q > 0 ? max_seqlen_q : 0);
  size_t n = align256((size_t)batch * hq * sq * sizeof(float));            // delta
  if (dtype != DH_F32) n += 2 * align256((size_t)batch * hq * ((sq + 31) / 32 * 32) * sizeof(float));
  if (dtype != DH_F32 && hk > 0 && hq / hk > 1)
    n += 2 * align256((size_t)(hq / hk) * (size_t)total_k * hk * d * sizeof(float));
  return n + 256;                                                          // the base pointer is rounded up to 256
}

}  // namespace dh

extern "C" void dh_attn_bwd_set_ds_limit(size_t bytes) { dh::g_ds_limit.store(bytes); }
extern "C" void dh_attn_bwd_set_ds_when_full(int on) { dh::g_ds_when_full.store(on ? 1 : 0); }

extern "C" size_t dh_attn_bwd_min_workspace_bytes(int64_t total_q, int64_t total_k, int batch, int max_seqlen_q, int hq,
                                                  int hk, int d, int dtype) {
  (void)total_q;
  return dh::bwd_base_bytes(total_k, batch, max_seqlen_q, hq, hk, d, dtype);
}

extern "C" size_t dh_attn_bwd_workspace_bytes(int64_t total_q, int64_t total_k, int batch, int max_seqlen_q, int hq,
                                              int hk, int d, int dtype) {
  using namespace dh;
  (void)total_q;
  // dS blocks, if a call of these sizes may keep them (causal or not is not known here: the causal grid is the smaller
  // one; the longest sequence has at most total_k keys)
  return bwd_base_bytes(total_k, batch, max_seqlen_q, hq, hk, d, dtype) +
         align256(ds_bytes(batch, max_seqlen_q, total_k, hq, d, dtype, 1));
}

extern "C" int dh_attn_bwd_one_launch(int batch, int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk,
                                      int d, int causal) {
  return dh::attn_bwd_route(batch, max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, causal, false).both ? 1 : 0;
}

// The route of a 16-bit call with a workspace of so many bytes.
static dh::AttnBwdRoute bwd_route_in(int batch, int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                                     int causal, size_t workspace_bytes) {
  using namespace dh;
  const size_t base = bwd_base_bytes(total_k, batch, max_seqlen_q, hq, hk, d, DH_BF16);
  const size_t dsb = ds_bytes(batch, max_seqlen_q, total_k, hq, d, DH_BF16, causal);
  return attn_bwd_route(batch, max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, causal, dsb > 0 && base + align256(dsb) <= workspace_bytes);
}

extern "C" int dh_attn_bwd_path(int batch, int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                                int causal, size_t workspace_bytes) {
  const dh::AttnBwdRoute r = bwd_route_in(batch, max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, causal, workspace_bytes);
  return (r.hand_dkv ? 1 : 0) | (r.keep_ds ? 2 : (r.hand_dq ? 4 : 0) | (r.big_dq ? 8 : 0));
}

extern "C" int dh_attn_bwd_dq_rows(int batch, int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                                   int causal, size_t workspace_bytes) {
  const dh::AttnBwdRoute r = bwd_route_in(batch, max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, causal, workspace_bytes);
  return r.keep_ds ? 0 : r.dq_rows;
}

static int attn_bwd_entry(const void *dout, const void *q, const void *k, const void *v, const void *out,
                          const float *lse, void *dq, void *dk, void *dv, float *delta_out, void *workspace,
                          size_t workspace_bytes, const int32_t *cu_seqlens_q, const int32_t *cu_seqlens_k, int batch,
                          int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                          int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                          int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride,
                          float softmax_scale, int causal, int dq_accumulate, int q_shift, int k_shift, int lse_pitch, int dtype,
                          void *stream) {
  using namespace dh;
  DH_CHECK(batch >= 0 && max_seqlen_q >= 0 && max_seqlen_k >= 0 && total_q >= 0 && total_k >= 0, "negative size");
  DH_CHECK(hq > 0 && hk > 0 && hq % hk == 0, "hq=%d must be a positive multiple of hk=%d", hq, hk);
  if (batch == 0) return DH_OK;
  DH_CHECK(dout && q && k && v && out && lse && dq && dk && dv && workspace && cu_seqlens_q && cu_seqlens_k,
           "null pointer");
  DH_CHECK(aligned16(workspace), "workspace must be 16-byte aligned");
  const size_t base_bytes = bwd_base_bytes(total_k, batch, max_seqlen_q, hq, hk, d, dtype);
  DH_CHECK(workspace_bytes >= base_bytes, "workspace of %zu bytes is smaller than the %zu bytes this call needs "
           "(dh_attn_bwd_min_workspace_bytes)", workspace_bytes, base_bytes);
  hipStream_t st = (hipStream_t)stream;
  uint8_t *ws = (uint8_t *)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  const size_t plane = align256((size_t)batch * hq * max_seqlen_q * sizeof(float));
  float *delta = delta_out ? delta_out : (float *)ws;
  ws += plane;
  float *ld2 = nullptr;
  const int ld2_pitch = (max_seqlen_q + 31) / 32 * 32;
  const size_t plane2 = align256((size_t)batch * hq * (size_t)ld2_pitch * sizeof(float));
  if (dtype != DH_F32) {
    ld2 = (float *)ws;
    ws += 2 * plane2;
    DH_CHECK(d != 128 || plane2 < (1ull << 31), "batch * heads * max_seqlen_q too large");
  }

  const int n = 16 / (int)dtype_size(dtype);
  DH_CHECK(d % n == 0 || dtype == DH_F32, "head dim %d must be a multiple of %d", d, n);
  DH_CHECK(do_stride % n == 0 && o_stride % n == 0 && aligned16(dout) && aligned16(out),
           "dout/out rows must be 16-byte aligned");
  // head dim 128 in 16 bits, two ways: with room for dS in the workspace the dK/dV kernel keeps it and dQ is one
  // product over it (delta from the delta kernel, which runs first); otherwise the dQ kernel recomputes S and dP,
  // forms delta itself and runs first.  fp32 uses the delta kernel.
  // dS is kept only if the blocks fit behind everything else in the workspace THIS call was given (and under the
  // process-wide limit); they take the tail of the workspace
  size_t dsb = ds_bytes(batch, max_seqlen_q, total_k, hq, d, dtype, causal);
  if (dsb > 0 && base_bytes + align256(dsb) > workspace_bytes) dsb = 0;
  const AttnBwdRoute route = attn_bwd_route(batch, max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, causal, dsb > 0,
                                            std::max({q_stride, k_stride, v_stride, do_stride, o_stride}) > ROWS_MAX_STRIDE / 2);
  uint8_t *ds_ws = (uint8_t *)(((uintptr_t)workspace + 255) & ~(uintptr_t)255) + (base_bytes - 256);
  const bool delta_in_dq = dtype != DH_F32 && !route.keep_ds;
  if (max_seqlen_q > 0 && !delta_in_dq) {
    DH_DISPATCH_DTYPE(dtype, {
      launch_delta<T>(dout, out, delta, lse, ld2, (int64_t)(plane2 / sizeof(float)), ld2_pitch, cu_seqlens_q, q_shift, lse_pitch,
                      batch, max_seqlen_q, hq, d, do_stride, o_stride, delta_out ? 1 : 0, st);
    });
  }
  if (dtype == DH_F32) {
    DH_CHECK(d > 0 && d <= 256 && d % 4 == 0, "fp32 attention needs d %% 4 == 0 and d <= 256 (got %d)", d);
    return attn_bwd_f32(dout, q, k, v, lse, delta, dq, dk, dv, cu_seqlens_q, cu_seqlens_k, batch, max_seqlen_q,
                        max_seqlen_k, hq, hk, d, q_stride, k_stride, v_stride, do_stride, dq_stride, dk_stride,
                        dv_stride, softmax_scale, causal, dq_accumulate, st);
  }
  DH_CHECK(d == 64 || d == 96 || d == 128 || d == 192 || d == 256,
           "bf16/fp16 attention supports head dims 64, 96, 128, 192 and 256 (got %d); pad other sizes with zero columns", d);
  DH_CHECK(q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && dq_stride % 4 == 0 && dk_stride % 4 == 0 &&
               dv_stride % 4 == 0,
           "token strides must keep rows aligned");
  DH_CHECK(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(dq) && aligned16(dk) && aligned16(dv),
           "pointers must be 16-byte aligned");
  AttnBwdParams p;
  p.dout = dout; p.q = q; p.k = k; p.v = v; p.lse = lse; p.delta = delta;
  p.out = out; p.o_stride = o_stride;
  p.ld2 = ld2; p.ld2_plane = (int64_t)(plane2 / sizeof(float)); p.ld2_pitch = ld2_pitch;
  p.dq = dq; p.dk = dk; p.dv = dv;
  p.cu_q = cu_seqlens_q; p.cu_k = cu_seqlens_k;
  p.max_sq = max_seqlen_q; p.hq = hq; p.hk = hk;
  p.total_k = total_k;
  p.q_stride = q_stride; p.k_stride = k_stride; p.v_stride = v_stride; p.do_stride = do_stride;
  p.dq_stride = dq_stride; p.dk_stride = dk_stride; p.dv_stride = dv_stride;
  p.scale = softmax_scale;
  p.scale_log2 = attn_scale_log2(softmax_scale);
  p.causal = causal;
  p.q_shift = q_shift; p.k_shift = k_shift; p.lse_pitch = lse_pitch;
  p.dq_accumulate = dq_accumulate ? 1 : 0;
  p.delta_tail = delta_out ? 1 : 0;
  p.ds = route.keep_ds ? (void *)ds_ws : nullptr;
  p.ds_nqt = 2 * (int)cdiv(max_seqlen_q, 64);
  p.ds_nkb = 2 * (int)cdiv(max_seqlen_k < total_k ? max_seqlen_k : total_k, 64) + 1;
  p.hsplit = route.hsplit;
  p.dk_part = nullptr;
  p.dv_part = nullptr;
  if (p.hsplit > 1) {
    const size_t part = align256((size_t)(hq / hk) * (size_t)total_k * hk * d * sizeof(float));
    p.dk_part = (float *)ws;
    p.dv_part = (float *)(ws + part);
  }
  DH_CHECK(k_stride < (1ll << 31) && v_stride < (1ll << 31) && q_stride < (1ll << 31) && do_stride < (1ll << 31),
           "token stride too large");
  int rc = DH_OK;
#define DH_BWD_D(TT)                                                                            \
  do {                                                                                          \
    const auto run = d == 64    ? bwd_passes<TT, 64>                                            \
                     : d == 96  ? bwd_passes<TT, 96>                                            \
                     : d == 128 ? bwd_passes<TT, 128>                                           \
                     : d == 192 ? bwd_passes<TT, 192>                                           \
                                : bwd_passes<TT, 256>;                                          \
    rc = run(p, route, batch, max_seqlen_q, max_seqlen_k, st);                                         \
  } while (0)
  if (dtype == DH_BF16) DH_BWD_D(bf16_t); else DH_BWD_D(f16_t);
#undef DH_BWD_D
  if (rc != DH_OK) return rc;
  DH_LAUNCH_CHECK();
  return DH_OK;
}

extern "C" int dh_attn_bwd(const void *dout, const void *q, const void *k, const void *v, const void *out,
                           const float *lse, void *dq, void *dk, void *dv, float *delta_out, void *workspace,
                           size_t workspace_bytes, const int32_t *cu_seqlens_q, const int32_t *cu_seqlens_k, int batch,
                           int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                           int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                           int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride,
                           float softmax_scale, int causal, int dtype, void *stream) {
  return attn_bwd_entry(dout, q, k, v, out, lse, dq, dk, dv, delta_out, workspace, workspace_bytes, cu_seqlens_q, cu_seqlens_k, batch,
                        max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, q_stride, k_stride, v_stride, o_stride,
                        do_stride, dq_stride, dk_stride, dv_stride, softmax_scale, causal, 0, 0, 0, max_seqlen_q, dtype, stream);
}

extern "C" int dh_attn_bwd_acc(const void *dout, const void *q, const void *k, const void *v, const void *out,
                               const float *lse, void *dq, void *dk, void *dv, float *delta_out, void *workspace,
                               size_t workspace_bytes, const int32_t *cu_seqlens_q, const int32_t *cu_seqlens_k,
                               int batch, int max_seqlen_q, int max_seqlen_k, int64_t total_q, int64_t total_k, int hq,
                               int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                               int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride,
                               float softmax_scale, int causal, int accumulate_dq, int dtype, void *stream) {
  return attn_bwd_entry(dout, q, k, v, out, lse, dq, dk, dv, delta_out, workspace, workspace_bytes, cu_seqlens_q, cu_seqlens_k, batch,
                        max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, q_stride, k_stride, v_stride, o_stride,
                        do_stride, dq_stride, dk_stride, dv_stride, softmax_scale, causal, accumulate_dq, 0, 0, max_seqlen_q, dtype, stream);
}

extern "C" int dh_attn_bwd_halves(const void *dout, const void *q, const void *k, const void *v, const void *out,
                                  const float *lse, void *dq, void *dk, void *dv, float *delta_out, void *workspace,
                                  size_t workspace_bytes, const int32_t *cu_seqlens_q, const int32_t *cu_seqlens_k,
                                  int q_shift, int k_shift, int lse_pitch, int batch, int max_seqlen_q,
                                  int max_seqlen_k, int64_t total_q, int64_t total_k, int hq, int hk, int d,
                                  int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                                  int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride,
                                  float softmax_scale, int causal, int accumulate_dq, int dtype, void *stream) {
  DH_CHECK((q_shift == 0 || q_shift == 1) && (k_shift == 0 || k_shift == 1), "sequences are taken whole or halved");
  DH_CHECK(dtype != DH_F32 || (q_shift + k_shift == 0 && lse_pitch == max_seqlen_q), "fp32 attention takes whole sequences");
  DH_CHECK(lse_pitch >= max_seqlen_q, "lse rows are shorter than max_seqlen_q");
  return attn_bwd_entry(dout, q, k, v, out, lse, dq, dk, dv, delta_out, workspace, workspace_bytes, cu_seqlens_q, cu_seqlens_k, batch,
                        max_seqlen_q, max_seqlen_k, total_q, total_k, hq, hk, d, q_stride, k_stride, v_stride, o_stride,
                        do_stride, dq_stride, dk_stride, dv_stride, softmax_scale, causal, accumulate_dq, q_shift, k_shift,
                        lse_pitch, dtype, stream);
}
