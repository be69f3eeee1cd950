// Attention forward on the tile layout of attn_tile.h (16 bits).  A workgroup is RG row groups (32 query rows each) x SPLIT
// key splits; an iteration has SPLIT tiles of BN keys (K and V) in LDS, split s works on tile it * SPLIT + s, and the tiles of
// the next iteration are copied global -> LDS meanwhile (two stages).  S^T = K Q^T puts a query row on each lane, P^T goes
// straight back in as the operand of O^T += V^T P^T; the splits' (O, m, l) are merged through LDS in split order.
//
// What bounds it: a 32 x 32 score block is D / 8 matrix instructions (D / 8 x 32 cycles) and about 100 vector instructions of
// softmax (400 cycles and more), so at head dim 64 the vector unit, at all of them the issue rate of the few wavefronts that
// fit, and for short sequences the chain of one wavefront.  Head dims 64 and 96 therefore fit 128 registers: two
// workgroups, 16 wavefronts, on a compute unit, whose matrix, softmax and LDS phases fill each other's waits without
// hand-written ordering (WPS: wavefronts per SIMD).  The 128-row form at head dim 256 does not fit its 256 registers: 12 are
// spilled (52 bytes a lane), read back by 5 loads in the loop.
// Measured against the register-staged kernels that these head dims ran before, forward, causal: 16 heads x 2 x 512,
// head dim 64 15.5 -> 9.4 us; 32 query / 8 kv heads x 4096, head dim 64 192 -> 94, 96 272 -> 132, 256 910 -> 329 us; 16
// heads x 2048, head dim 192 324 -> 56 us.  With the wait for Q in front of the loop (loaded_here): 16 x 2 x 512 10.0 -> 8.5 us
// with its launch, 16 x 1024 12.5 -> 11.1, head dim 192 32 -> 29.5 us.
#include "attn_tile.h"

namespace dh {

template <typename T, int D, int RG, int SPLIT, int BN, int WPS>
__global__ void __launch_bounds__(64 * RG * SPLIT, WPS) attn_fwd_tile_kernel(const AttnFwdParams p) {
  using M = Mma<T>;
  using Frag = typename M::Frag;
  using A = AttnTile<D>;
  constexpr int BM = 32 * RG, NB = BN / 32, NS = BN / 16, NW = RG * SPLIT;
  constexpr int TILEB = BN * D * (int)sizeof(T);          // bytes of one K (or V) tile
  constexpr int STAGEB = SPLIT * 2 * TILEB;               // K tiles of all splits, then V tiles
  constexpr int RPW = SPLIT * 2 * BN / NW;                // rows that a wavefront copies per iteration
  constexpr int SLOTF = 32 * D;                           // floats of a wavefront's O
  constexpr int EXB = (SPLIT - 1) * RG * (SLOTF + 128) * 4;
  static_assert(RPW % 16 == 0 && RPW <= BN, "whole copy patterns of one tile per wavefront");
  __shared__ __attribute__((aligned(1024))) char sAll[2 * STAGEB > EXB ? 2 * STAGEB : EXB];

  rng_state_zero(p);
  const int b = seq_by_length(p.cu_q, gridDim.y, blockIdx.y);
  // the query heads of one kv head read the same K / V rows: keep a kv head on one XCD's L2, late causal tiles first
  const int ratio = p.hq / p.hk, P = gridDim.x / p.hq;
  int hkv, item;
  xcd_group_item(blockIdx.x, p.hk, ratio * P, hkv, item);
  const int h = hkv * ratio + item % ratio, px = item / ratio;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nqt = (sq + BM - 1) / BM;
  if (px >= nqt) return;
  const int m0 = (nqt - 1 - px) * BM;
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

  const int wrow0 = m0 + rg * 32, row_q = wrow0 + c;
  const int row_ld = row_q < sq ? row_q : sq - 1;
  const T *qp = reinterpret_cast<const T *>(p.q) + (int64_t)(q0 + row_ld) * p.q_stride + (int64_t)h * D;
  Frag Qf[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) Qf[ks] = frag_ld<T>(qp + ks * 16 + 8 * hh);
  const RowLane rl = row_lane<D>(lane);
  const TrLane tl = tr_lane<D>(lane);

  int nk_end = sk;
  if (causal && m0 + BM < nk_end) nk_end = m0 + BM;
  const int ntiles = (nk_end + BN - 1) / BN;
  const int niter = (ntiles + SPLIT - 1) / SPLIT;

  floatx16 O[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) O[t][v] = 0.f;
  float m_run = -1e30f, l_run = 0.f;

  auto issue = [&](int it) {
    const int tile = it * SPLIT + cp_sp;
    if (tile < ntiles) copy_tile<T, D, RPW>(cp_g, cp_stride, tile * BN + cp_r0, sk, cp_whole, cp_dst + (uint32_t)((it & 1) * STAGEB), cl, lane);
  };
  if (niter > 0) issue(0);
  if constexpr (D < 256 || RG == 2) loaded_here(Qf);        // (more of them would be spilled in the 128-row form at 256)
#pragma unroll 1
  for (int it = 0; it < niter; ++it) {
    dma_wait_all();
    __syncthreads();   // this stage has landed, and everyone is done with the other one
    if (it + 1 < niter) issue(it + 1);
    const int tile = it * SPLIT + sp, n0 = tile * BN;
    if (tile < ntiles && !(causal && n0 > wrow0 + 31)) {
      const uint32_t kt = lds0 + (uint32_t)((it & 1) * STAGEB + sp * TILEB), vt = kt + (uint32_t)(SPLIT * TILEB);
      floatx16 S[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) S[nb][v] = 0.f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) S[nb] = M::mma(row_frag<T, D>(kt + (uint32_t)(nb * 32 * A::PITCH), rl, ks), Qf[ks], S[nb]);
      if ((causal && n0 + BN - 1 > wrow0) || n0 + BN > sk) {
        const int lim = causal && row_q + 1 < sk ? row_q + 1 : sk;        // keys this lane's row attends to
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int v = 0; v < 16; ++v) S[nb][v] = n0 + nb * 32 + acc_row(v, hh) < lim ? S[nb][v] : -INFINITY;
      }
      float mx = S[0][0];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, S[nb][v]);
      // the running maximum is only a reference point: it moves when some row has grown past it by more than
      // DH_FWD_RESCALE_LOG2 binades (see the head-dim-128 kernel)
      const float m_new = fmaxf(m_run, pair32_max(mx));
      if (__any((m_new - m_run) * scale_log2 > (float)DH_FWD_RESCALE_LOG2)) {
        const float alpha = fast_exp2((m_run - m_new) * scale_log2);
        l_run *= alpha;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) O[t][v] *= alpha;
        m_run = m_new;
      }
      const float mc = m_run * scale_log2;
      float ps = 0.f;
      Frag Pb[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        float pv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          pv[j] = fast_exp2(S[s >> 1][8 * (s & 1) + j] * scale_log2 - mc);
          ps += pv[j];
        }
        Pb[s] = frag_pack<T>(pv);
      }
      l_run += ps;
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
          O[t] = M::mma(tr_frag<T, D>(vt, tl, t, s), Pb[s], O[t]);
    }
  }
  __syncthreads();

  // merge the splits: slot x = (split - 1) * RG + row group holds O, the m and l planes follow the slots
  float *xo = reinterpret_cast<float *>(sAll), *xml = xo + (SPLIT - 1) * RG * SLOTF;
  if (sp > 0) {
    const int x = (sp - 1) * RG + rg;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) xo[x * SLOTF + (t * 16 + v) * 64 + lane] = O[t][v];
    xml[x * 128 + lane] = m_run;
    xml[x * 128 + 64 + lane] = l_run;
  }
  __syncthreads();
  if (sp > 0) return;
#pragma unroll
  for (int s2 = 1; s2 < SPLIT; ++s2) {
    const int x = (s2 - 1) * RG + rg;
    const float m_o = xml[x * 128 + lane], l_o = xml[x * 128 + 64 + lane];
    const float m_new = fmaxf(m_run, m_o);
    const float a_me = fast_exp2((m_run - m_new) * scale_log2), a_o = fast_exp2((m_o - m_new) * scale_log2);
    l_run = l_run * a_me + l_o * a_o;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) O[t][v] = O[t][v] * a_me + xo[x * SLOTF + (t * 16 + v) * 64 + lane] * a_o;
    m_run = m_new;
  }
  const float l_tot = pair32_sum(l_run);
  const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  if (row_q < sq) {
    T *op = reinterpret_cast<T *>(p.o) + (int64_t)(q0 + row_q) * p.o_stride + (int64_t)h * D;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int vb = 0; vb < 4; ++vb) {
        Quad<T> o4;
#pragma unroll
        for (int j = 0; j < 4; ++j) o4.v[j] = static_cast<T>(O[t][4 * vb + j] * inv);
        *reinterpret_cast<Quad<T> *>(op + 32 * t + 8 * vb + 4 * hh) = o4;
      }
    if (hh == 0) p.lse[((int64_t)b * p.hq + h) * p.max_sq + row_q] = l_tot > 0.f ? m_run * p.scale + logf(l_tot) : -INFINITY;
  }
}

template <typename T, int D, int RG, int SPLIT, int BN, int WPS>
static int launch_attn_fwd_tile(const AttnFwdParams &p, int batch, hipStream_t st) {
  dim3 grid((unsigned)(cdiv(p.max_sq, 32 * RG) * p.hq), (unsigned)batch);
  hipLaunchKernelGGL((attn_fwd_tile_kernel<T, D, RG, SPLIT, BN, WPS>), grid, dim3(64 * RG * SPLIT), 0, st, p);
  return DH_OK;
}

}  // namespace dh
