// fp32 attention forward / backward (exact fp32 arithmetic: v_mfma_f32_32x32x2_f32 and expf).
//
// Head dims up to 128: one wavefront owns 32 query rows (forward, dQ) or 32 key rows (dK/dV) and walks tiles of 32 rows
// of the other sequence; four wavefronts of a workgroup share the owned rows and split the tiles (tile it * 4 + w), and
// their partial results are added in wavefront order through LDS at the end (deterministic).  The layouts are those of
// the 16-bit kernels: S^T = K Q^T puts a query row on each lane, and an accumulator goes straight back in as the next
// product's operand.  For the fp32 instruction (one k per lane half) this makes both reads of a matrix plain loads:
//   * row fragments (the operand whose contraction runs along d): a lane reads 4 floats at k = 8 i + 4 h, which are the
//     operands of four instructions with k = {8 i + j, 8 i + 4 + j};
//   * column fragments (contraction along the rows): instruction v takes row 8 (v / 4) + 4 h + v % 4 and lane c the
//     columns N c .. N c + N - 1 (N = D / 32), one contiguous 128 N byte run per half wavefront.
// Nothing is shared between wavefronts, so operands go from the caches to registers with no LDS stage and no barrier
// in the loop; each operand's loads for the next tile are issued right after its last use.
//
// What bounds it: at the small parity layer (2 x 512 rows, 16 heads of 64) the chain of one wavefront.  One workgroup
// per row without matrix cores, the form kept below for head dims above 128, walks the other sequence's rows one
// 4-byte column load at a time: forward / dQ / dKdV took 224 / 307 / 578 us that way and take 31 / 44 / 60 us here (7 / 11 / 15 us of matrix time).
#include "mma.h"

namespace dh {

// ---- head dims up to 128: matrix cores ---------------------------------------------------------------------------
constexpr int FS = 4;           // wavefronts of a workgroup = splits of the walked sequence

__device__ __forceinline__ floatx16 mma_f32(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4u __attribute__((aligned(4)));

// Row fragments of one row: D / 8 pieces of 4 floats at 8 i + 4 h.  FULL: d == D; else zeros from column d on (the load
// itself is never predicated: it goes to column 0 instead).
template <int D, bool FULL> __device__ __forceinline__ void rows_load(f32x4 (&f)[D / 8], const float *row, int hh, int d) {
#pragma unroll
  for (int i = 0; i < D / 8; ++i) {
    const int c = 8 * i + 4 * hh;
    const bool in = FULL || c < d;
    const f32x4 x = *reinterpret_cast<const f32x4 *>(row + (in ? c : 0));
    f[i] = in ? x : (f32x4)(0.f);
  }
}

template <int N> struct FVec { typedef float V __attribute__((ext_vector_type(N))); };

// Column fragments of a 32-row tile starting at row0 (rows clamped to the last one): f[v] holds columns N c .. of row
// 8 (v / 4) + 4 h + v % 4.  A tile inside the sequence is addressed as wave-uniform row base + one lane offset.
template <int D, bool FULL> __device__ __forceinline__ void cols_load(typename FVec<D / 32>::V (&f)[16], const float *base,
                                                                      int64_t stride, int row0, int rows, int c, int hh, int d) {
  constexpr int N = D / 32;
  using V = typename FVec<N>::V;
  const bool in = FULL || N * c < d;
  const int col = in ? N * c : 0;
  if (row0 + 32 <= rows) {
    const int lane_off = 4 * hh * (int)stride + col;
#pragma unroll
    for (int v = 0; v < 16; ++v)
      f[v] = *reinterpret_cast<const V *>(base + (int64_t)(row0 + acc_row(v, 0)) * stride + lane_off);
  } else {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      int r = row0 + acc_row(v, hh);
      r = r < rows ? r : rows - 1;
      f[v] = *reinterpret_cast<const V *>(base + (int64_t)r * stride + col);
    }
  }
  if (!FULL) {
#pragma unroll
    for (int v = 0; v < 16; ++v) f[v] = in ? f[v] : (V)(0.f);
  }
}

// acc = A B^T over d from row fragments.
template <int D> __device__ __forceinline__ floatx16 rows_product(const f32x4 (&a)[D / 8], const f32x4 (&b)[D / 8]) {
  floatx16 s;
#pragma unroll
  for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
  for (int i = 0; i < D / 8; ++i) {
    s = mma_f32(a[i].x, b[i].x, s);
    s = mma_f32(a[i].y, b[i].y, s);
    s = mma_f32(a[i].z, b[i].z, s);
    s = mma_f32(a[i].w, b[i].w, s);
  }
  return s;
}

// acc[t] += X^T P over the tile's rows: X in column fragments, P an accumulator.
template <int N> __device__ __forceinline__ void cols_product(floatx16 (&acc)[N], const typename FVec<N>::V (&x)[16], const floatx16 &p) {
#pragma unroll
  for (int v = 0; v < 16; ++v) {
#pragma unroll
    for (int t = 0; t < N; ++t) acc[t] = mma_f32(x[v][t], p[v], acc[t]);
  }
}

// This wavefront's accumulators (owned row c on lanes, d = N acc_row + t) as rows of D + 4 floats in LDS.
template <int D> __device__ __forceinline__ void acc_to_lds(float *dst, const floatx16 (&acc)[D / 32], float mul, int c, int hh) {
  constexpr int N = D / 32;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    typename FVec<N>::V x;
#pragma unroll
    for (int t = 0; t < N; ++t) x[t] = acc[t][v] * mul;
    *reinterpret_cast<typename FVec<N>::V *>(dst + c * (D + 4) + N * acc_row(v, hh)) = x;
  }
}

// The workgroup's FS partial blocks added in order, times mul, to rows row0 .. of `out` (added to what is there if add).
template <int D> __device__ __forceinline__ void lds_sum_store(const float *part, float *out, int64_t stride, int row0, int rows,
                                                               int d, float mul, bool add) {
  for (int i = threadIdx.x; i < 32 * (D / 4); i += 64 * FS) {
    const int r = i / (D / 4), c = 4 * (i % (D / 4));
    if (row0 + r >= rows || c >= d) continue;
    float4 s = *reinterpret_cast<const float4 *>(part + r * (D + 4) + c);
#pragma unroll
    for (int w = 1; w < FS; ++w) {
      const float4 x = *reinterpret_cast<const float4 *>(part + (w * 32 + r) * (D + 4) + c);
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    float4 *o = reinterpret_cast<float4 *>(out + (int64_t)(row0 + r) * stride + c);
    s.x *= mul; s.y *= mul; s.z *= mul; s.w *= mul;
    if (add) {
      const float4 x = *o;
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    *o = s;
  }
}

template <int D> constexpr int f32_lds_bytes() { return FS * 32 * (D + 4) * 4; }

template <int D, bool FULL>
__global__ void __launch_bounds__(64 * FS)
attn_fwd_f32_mma_kernel(const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
                        float *__restrict__ out, float *__restrict__ lse, const int32_t *__restrict__ cu_q,
                        const int32_t *__restrict__ cu_k, int max_sq, int hq, int hk, int d, int64_t q_stride,
                        int64_t k_stride, int64_t v_stride, int64_t o_stride, float scale, int causal) {
  constexpr int N = D / 32;
  extern __shared__ __attribute__((aligned(16))) float f32_lds[];
  __shared__ float sm[FS][32], sl[FS][32];
  const int b = blockIdx.z, h = blockIdx.y;
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  const int m0 = 32 * (int)(gridDim.x - 1 - blockIdx.x);      // late causal tiles carry the most work and come first
  if (m0 >= sq) return;
  const int hkv = h / (hq / hk);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int row_q = m0 + c, row_ld = row_q < sq ? row_q : sq - 1;
  const float *kg = k + (int64_t)k0 * k_stride + (int64_t)hkv * d;
  const float *vg = v + (int64_t)k0 * v_stride + (int64_t)hkv * d;
  const int nk = causal && m0 + 32 < sk ? m0 + 32 : sk;
  const int nt = (nk + 31) / 32;
  const int k_lim = causal && row_q + 1 < sk ? row_q + 1 : sk;        // keys this lane's row attends to

  f32x4 Q[D / 8], K[D / 8];
  typename FVec<N>::V V[16];
  floatx16 O[N];
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int x = 0; x < 16; ++x) O[t][x] = 0.f;
  float m_run = -1e30f, l_run = 0.f;
  rows_load<D, FULL>(Q, q + (int64_t)(q0 + row_ld) * q_stride + (int64_t)h * d, hh, d);
  auto load_k = [&](int n0) {
    const int r = n0 + c < sk ? n0 + c : sk - 1;
    rows_load<D, FULL>(K, kg + (int64_t)r * k_stride, hh, d);
  };
  if (w < nt) {
    load_k(32 * w);
    cols_load<D, FULL>(V, vg, v_stride, 32 * w, sk, c, hh, d);
  }
  for (int it = w; it < nt; it += FS) {
    const int n0 = 32 * it, nn = it + FS < nt ? n0 + 32 * FS : n0;     // the last trip loads its own tile again, unused
    floatx16 S = rows_product<D>(K, Q);
    load_k(nn);
    const bool mask = (causal && n0 + 31 > m0) || n0 + 32 > sk;
    float mx = -INFINITY;
#pragma unroll
    for (int x = 0; x < 16; ++x) S[x] *= scale;
    if (mask) {
#pragma unroll
      for (int x = 0; x < 16; ++x) S[x] = n0 + acc_row(x, hh) < k_lim ? S[x] : -INFINITY;
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) mx = fmaxf(mx, S[x]);
    const float m_new = fmaxf(m_run, pair32_max(mx));
    if (__any(m_new > m_run)) {
      const float alpha = expf(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int t = 0; t < N; ++t)
#pragma unroll
        for (int x = 0; x < 16; ++x) O[t][x] *= alpha;
      m_run = m_new;
    }
    float ps = 0.f;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      S[x] = expf(S[x] - m_new);
      ps += S[x];
    }
    l_run += ps;
    cols_product<N>(O, V, S);
    cols_load<D, FULL>(V, vg, v_stride, nn, sk, c, hh, d);
  }
  // the splits' (O, m, l) become one
  l_run = pair32_sum(l_run);
  if (hh == 0) {
    sm[w][c] = m_run;
    sl[w][c] = l_run;
  }
  __syncthreads();
  float m = sm[0][c], l = 0.f;
#pragma unroll
  for (int x = 1; x < FS; ++x) m = fmaxf(m, sm[x][c]);
#pragma unroll
  for (int x = 0; x < FS; ++x) l += sl[x][c] * expf(sm[x][c] - m);
  acc_to_lds<D>(f32_lds + w * 32 * (D + 4), O, l > 0.f ? expf(m_run - m) / l : 0.f, c, hh);
  if (w == 0 && hh == 0 && row_q < sq) lse[((int64_t)b * hq + h) * max_sq + row_q] = l > 0.f ? m + logf(l) : -INFINITY;
  __syncthreads();
  lds_sum_store<D>(f32_lds, out + (int64_t)q0 * o_stride + (int64_t)h * d, o_stride, m0, sq, d, 1.f, false);
}

template <int D, bool FULL>
__global__ void __launch_bounds__(64 * FS)
attn_bwd_dq_f32_mma_kernel(const float *__restrict__ dout, const float *__restrict__ q, const float *__restrict__ k,
                           const float *__restrict__ v, const float *__restrict__ lse, const float *__restrict__ delta,
                           float *__restrict__ dq, const int32_t *__restrict__ cu_q, const int32_t *__restrict__ cu_k,
                           int max_sq, int hq, int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                           int64_t do_stride, int64_t dq_stride, float scale, int causal, int accumulate) {
  constexpr int N = D / 32;
  extern __shared__ __attribute__((aligned(16))) float f32_lds[];
  const int b = blockIdx.z, h = blockIdx.y;
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  const int m0 = 32 * (int)(gridDim.x - 1 - blockIdx.x);
  if (m0 >= sq) return;
  const int hkv = h / (hq / hk);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int row_q = m0 + c, row_ld = row_q < sq ? row_q : sq - 1;
  const float *kg = k + (int64_t)k0 * k_stride + (int64_t)hkv * d;
  const float *vg = v + (int64_t)k0 * v_stride + (int64_t)hkv * d;
  const int nk = causal && m0 + 32 < sk ? m0 + 32 : sk;
  const int nt = (nk + 31) / 32;
  const int k_lim = causal && row_q + 1 < sk ? row_q + 1 : sk;        // keys this lane's row attends to

  f32x4 Q[D / 8], dO[D / 8], K[D / 8], V[D / 8];
  typename FVec<N>::V Kc[16];
  floatx16 acc[N];
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[t][x] = 0.f;
  rows_load<D, FULL>(Q, q + (int64_t)(q0 + row_ld) * q_stride + (int64_t)h * d, hh, d);
  rows_load<D, FULL>(dO, dout + (int64_t)(q0 + row_ld) * do_stride + (int64_t)h * d, hh, d);
  const float li = lse[((int64_t)b * hq + h) * max_sq + row_ld];
  const float di = delta[((int64_t)b * hq + h) * max_sq + row_ld];
  auto load_rows = [&](int n0) {
    const int r = n0 + c < sk ? n0 + c : sk - 1;
    rows_load<D, FULL>(K, kg + (int64_t)r * k_stride, hh, d);
    rows_load<D, FULL>(V, vg + (int64_t)r * v_stride, hh, d);
  };
  if (w < nt) {
    load_rows(32 * w);
    cols_load<D, FULL>(Kc, kg, k_stride, 32 * w, sk, c, hh, d);
  }
  for (int it = w; it < nt; it += FS) {
    const int n0 = 32 * it, nn = it + FS < nt ? n0 + 32 * FS : n0;
    floatx16 S = rows_product<D>(K, Q);
    const floatx16 dP = rows_product<D>(V, dO);
    load_rows(nn);
    const bool mask = (causal && n0 + 31 > m0) || n0 + 32 > sk;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const float pj = expf(S[x] * scale - li);
      S[x] = pj * (dP[x] - di);
    }
    if (mask) {
#pragma unroll
      for (int x = 0; x < 16; ++x) S[x] = n0 + acc_row(x, hh) < k_lim ? S[x] : 0.f;
    }
    cols_product<N>(acc, Kc, S);
    cols_load<D, FULL>(Kc, kg, k_stride, nn, sk, c, hh, d);
  }
  acc_to_lds<D>(f32_lds + w * 32 * (D + 4), acc, 1.f, c, hh);
  __syncthreads();
  lds_sum_store<D>(f32_lds, dq + (int64_t)q0 * dq_stride + (int64_t)h * d, dq_stride, m0, sq, d, scale, accumulate != 0);
}

template <int D, bool FULL>
__global__ void __launch_bounds__(64 * FS)
attn_bwd_dkv_f32_mma_kernel(const float *__restrict__ dout, const float *__restrict__ q, const float *__restrict__ k,
                            const float *__restrict__ v, const float *__restrict__ lse, const float *__restrict__ delta,
                            float *__restrict__ dk, float *__restrict__ dv, const int32_t *__restrict__ cu_q,
                            const int32_t *__restrict__ cu_k, int max_sq, int hq, int hk, int d, int64_t q_stride,
                            int64_t k_stride, int64_t v_stride, int64_t do_stride, int64_t dk_stride, int64_t dv_stride,
                            float scale, int causal) {
  constexpr int N = D / 32;
  extern __shared__ __attribute__((aligned(16))) float f32_lds[];
  const int b = blockIdx.z, hkv = blockIdx.y, j0 = 32 * blockIdx.x;      // early causal tiles carry the most work
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  if (j0 >= sk) return;
  const int ratio = hq / hk;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int row_k = j0 + c, row_ld = row_k < sk ? row_k : sk - 1;
  const int t_beg = causal ? j0 / 32 : 0, ntq = (sq + 31) / 32 - t_beg;      // query tiles of one head
  const int nt = ntq > 0 ? ntq * ratio : 0;
  const int i_lo = row_k >= sk ? sq : causal ? row_k : 0;        // first query row that attends to this lane's key

  f32x4 K[D / 8], V[D / 8], Q[D / 8], dO[D / 8];
  typename FVec<N>::V Qc[16], dOc[16];
  float L[16], Dl[16];
  floatx16 dK[N], dV[N];
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      dK[t][x] = 0.f;
      dV[t][x] = 0.f;
    }
  rows_load<D, FULL>(K, k + (int64_t)(k0 + row_ld) * k_stride + (int64_t)hkv * d, hh, d);
  rows_load<D, FULL>(V, v + (int64_t)(k0 + row_ld) * v_stride + (int64_t)hkv * d, hh, d);
  auto head_of = [&](int it) { return hkv * ratio + it / ntq; };
  auto row0_of = [&](int it) { return 32 * (t_beg + it % ntq); };
  auto load_rows = [&](int it) {
    const int h = head_of(it), i0 = row0_of(it);
    const int r = i0 + c < sq ? i0 + c : sq - 1;
    rows_load<D, FULL>(Q, q + (int64_t)(q0 + r) * q_stride + (int64_t)h * d, hh, d);
    rows_load<D, FULL>(dO, dout + (int64_t)(q0 + r) * do_stride + (int64_t)h * d, hh, d);
    const int64_t at = ((int64_t)b * hq + h) * max_sq;
    if (i0 + 32 <= sq) {
#pragma unroll
      for (int x = 0; x < 16; x += 4) {
        const f32x4u l4 = *reinterpret_cast<const f32x4u *>(lse + at + i0 + acc_row(x, hh));
        const f32x4u d4 = *reinterpret_cast<const f32x4u *>(delta + at + i0 + acc_row(x, hh));
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          L[x + y] = l4[y];
          Dl[x + y] = d4[y];
        }
      }
    } else {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        int i = i0 + acc_row(x, hh);
        i = i < sq ? i : sq - 1;
        L[x] = lse[at + i];
        Dl[x] = delta[at + i];
      }
    }
  };
  auto load_cols = [&](int it) {
    const int h = head_of(it), i0 = row0_of(it);
    cols_load<D, FULL>(dOc, dout + (int64_t)q0 * do_stride + (int64_t)h * d, do_stride, i0, sq, c, hh, d);
    cols_load<D, FULL>(Qc, q + (int64_t)q0 * q_stride + (int64_t)h * d, q_stride, i0, sq, c, hh, d);
  };
  // D = 128: the owned rows, both accumulators and one tile's fragments fill the registers; loads go out where they are
  // used.
  constexpr bool AHEAD = D <= 64;
  if (AHEAD && w < nt) {
    load_rows(w);
    load_cols(w);
  }
  for (int it = w; it < nt; it += FS) {
    const int i0 = row0_of(it), nx = it + FS < nt ? it + FS : it;
    if (!AHEAD) load_rows(it);
    floatx16 P = rows_product<D>(Q, K);
    floatx16 dS = rows_product<D>(dO, V);
    const bool mask = (causal && i0 < j0 + 31) || i0 + 32 > sq || j0 + 32 > sk;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const float pj = expf(P[x] * scale - L[x]);
      P[x] = pj;
      dS[x] = pj * (dS[x] - Dl[x]);
    }
    if (mask) {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const int i = i0 + acc_row(x, hh);
        const bool in = i >= i_lo && i < sq;
        P[x] = in ? P[x] : 0.f;
        dS[x] = in ? dS[x] : 0.f;
      }
    }
    if (AHEAD) load_rows(nx);
    else load_cols(it);
    cols_product<N>(dV, dOc, P);
    cols_product<N>(dK, Qc, dS);
    if (AHEAD) load_cols(nx);
  }
  acc_to_lds<D>(f32_lds + w * 32 * (D + 4), dV, 1.f, c, hh);
  __syncthreads();
  lds_sum_store<D>(f32_lds, dv + (int64_t)k0 * dv_stride + (int64_t)hkv * d, dv_stride, j0, sk, d, 1.f, false);
  __syncthreads();
  acc_to_lds<D>(f32_lds + w * 32 * (D + 4), dK, 1.f, c, hh);
  __syncthreads();
  lds_sum_store<D>(f32_lds, dk + (int64_t)k0 * dk_stride + (int64_t)hkv * d, dk_stride, j0, sk, d, scale, false);
}

template <int D, bool FULL>
int attn_fwd_f32_mma(const float *q, const float *k, const float *v, float *out, float *lse, const int32_t *cu_q,
                     const int32_t *cu_k, int batch, int max_sq, int hq, int hk, int d, int64_t q_stride, int64_t k_stride,
                     int64_t v_stride, int64_t o_stride, float scale, int causal, hipStream_t st) {
  DH_MAX_DYNAMIC_LDS_PER_DEVICE((attn_fwd_f32_mma_kernel<D, FULL>), f32_lds_bytes<D>());
  hipLaunchKernelGGL((attn_fwd_f32_mma_kernel<D, FULL>), dim3((unsigned)cdiv(max_sq, 32), (unsigned)hq, (unsigned)batch), dim3(64 * FS),
                     f32_lds_bytes<D>(), st, q, k, v, out, lse, cu_q, cu_k, max_sq, hq, hk, d, q_stride, k_stride, v_stride,
                     o_stride, scale, causal);
  DH_LAUNCH_CHECK();
  return DH_OK;
}

template <int D, bool FULL>
int attn_bwd_f32_mma(const float *dout, const float *q, const float *k, const float *v, const float *lse, const float *delta,
                     float *dq, float *dk, float *dv, const int32_t *cu_q, const int32_t *cu_k, int batch, int max_sq,
                     int max_sk, int hq, int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                     int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride, float scale, int causal,
                     int dq_accumulate, hipStream_t st) {
  DH_MAX_DYNAMIC_LDS_PER_DEVICE((attn_bwd_dq_f32_mma_kernel<D, FULL>), f32_lds_bytes<D>());
  DH_MAX_DYNAMIC_LDS_PER_DEVICE((attn_bwd_dkv_f32_mma_kernel<D, FULL>), f32_lds_bytes<D>());
  if (max_sq > 0)
    hipLaunchKernelGGL((attn_bwd_dq_f32_mma_kernel<D, FULL>), dim3((unsigned)cdiv(max_sq, 32), (unsigned)hq, (unsigned)batch),
                       dim3(64 * FS), f32_lds_bytes<D>(), st, dout, q, k, v, lse, delta, dq, cu_q, cu_k, max_sq, hq, hk, d,
                       q_stride, k_stride, v_stride, do_stride, dq_stride, scale, causal, dq_accumulate);
  if (max_sk > 0)
    hipLaunchKernelGGL((attn_bwd_dkv_f32_mma_kernel<D, FULL>), dim3((unsigned)cdiv(max_sk, 32), (unsigned)hk, (unsigned)batch),
                       dim3(64 * FS), f32_lds_bytes<D>(), st, dout, q, k, v, lse, delta, dk, dv, cu_q, cu_k, max_sq, hq, hk, d,
                       q_stride, k_stride, v_stride, do_stride, dk_stride, dv_stride, scale, causal);
  DH_LAUNCH_CHECK();
  return DH_OK;
}

// ---- head dims above 128: one workgroup of 128 threads owns one query row (forward, dQ) or one key/value row (dK/dV)
// and walks the other sequence in chunks of 128: each thread scores one row of the chunk, the probabilities go through
// LDS, and each thread then accumulates the output columns it owns, in a fixed order.  (The accumulators and operands of
// the kernels above do not fit the registers at these sizes.)
constexpr int F32_NT = 128;     // threads per block = rows per chunk
constexpr int F32_MAXC = 2;     // columns per thread (d <= 256)

__device__ __forceinline__ float block128_reduce(float v, float *red, bool is_max) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float u = __shfl_xor(v, o, 64);
    v = is_max ? fmaxf(v, u) : v + u;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return is_max ? fmaxf(red[0], red[1]) : red[0] + red[1];
}

__device__ __forceinline__ float dot_row(const float *a_lds, const float *__restrict__ b, int d) {
  float s = 0.f;
  for (int i = 0; i < d; i += 4) {
    const float4 x = *reinterpret_cast<const float4 *>(b + i);
    s += a_lds[i] * x.x + a_lds[i + 1] * x.y + a_lds[i + 2] * x.z + a_lds[i + 3] * x.w;
  }
  return s;
}

__global__ void __launch_bounds__(F32_NT)
attn_fwd_f32_kernel(const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
                    float *__restrict__ out, float *__restrict__ lse, const int32_t *__restrict__ cu_q,
                    const int32_t *__restrict__ cu_k, int max_sq, int hq, int hk, int d, int64_t q_stride,
                    int64_t k_stride, int64_t v_stride, int64_t o_stride, float scale, int causal) {
  __shared__ float sq_row[256];
  __shared__ float sp[F32_NT];
  __shared__ float red[2];
  const int b = blockIdx.z, h = blockIdx.y, i = blockIdx.x;
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  if (i >= sq) return;
  const int hkv = h / (hq / hk);
  const int tid = threadIdx.x;
  const float *qr = q + (int64_t)(q0 + i) * q_stride + (int64_t)h * d;
  for (int c = tid; c < d; c += F32_NT) sq_row[c] = qr[c];
  __syncthreads();
  const int kend = causal ? (i + 1 < sk ? i + 1 : sk) : sk;
  float m_run = -INFINITY, l_run = 0.f, acc[F32_MAXC] = {0.f, 0.f};
  for (int j0 = 0; j0 < kend; j0 += F32_NT) {
    const int j = j0 + tid;
    float s = -INFINITY;
    if (j < kend) s = scale * dot_row(sq_row, k + (int64_t)(k0 + j) * k_stride + (int64_t)hkv * d, d);
    const float m_new = fmaxf(m_run, block128_reduce(s, red, true));
    const float pj = j < kend ? expf(s - m_new) : 0.f;
    const float alpha = expf(m_run - m_new);  // 0 on the first chunk (m_run = -inf)
    const float psum = block128_reduce(pj, red, false);
    l_run = l_run * alpha + psum;
    m_run = m_new;
    sp[tid] = pj;
    __syncthreads();
    const int cnt = kend - j0 < F32_NT ? kend - j0 : F32_NT;
#pragma unroll
    for (int ci = 0; ci < F32_MAXC; ++ci) {
      const int c = tid + ci * F32_NT;
      if (c < d) {
        float a = acc[ci] * alpha;
        const float *vp = v + (int64_t)(k0 + j0) * v_stride + (int64_t)hkv * d + c;
        for (int jj = 0; jj < cnt; ++jj) a += sp[jj] * vp[(int64_t)jj * v_stride];
        acc[ci] = a;
      }
    }
    __syncthreads();
  }
  float *orow = out + (int64_t)(q0 + i) * o_stride + (int64_t)h * d;
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
#pragma unroll
  for (int ci = 0; ci < F32_MAXC; ++ci) {
    const int c = tid + ci * F32_NT;
    if (c < d) orow[c] = acc[ci] * inv;
  }
  if (tid == 0) lse[((int64_t)b * hq + h) * max_sq + i] = l_run > 0.f ? m_run + logf(l_run) : -INFINITY;
}

// dQ: one block per query row.
__global__ void __launch_bounds__(F32_NT)
attn_bwd_dq_f32_kernel(const float *__restrict__ dout, const float *__restrict__ q, const float *__restrict__ k,
                       const float *__restrict__ v, const float *__restrict__ lse, const float *__restrict__ delta,
                       float *__restrict__ dq, const int32_t *__restrict__ cu_q, const int32_t *__restrict__ cu_k,
                       int max_sq, int hq, int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                       int64_t do_stride, int64_t dq_stride, float scale, int causal, int accumulate) {
  __shared__ float sq_row[256], sdo_row[256];
  __shared__ float sds[F32_NT];
  const int b = blockIdx.z, h = blockIdx.y, i = blockIdx.x;
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  if (i >= sq) return;
  const int hkv = h / (hq / hk);
  const int tid = threadIdx.x;
  const float *qr = q + (int64_t)(q0 + i) * q_stride + (int64_t)h * d;
  const float *dor = dout + (int64_t)(q0 + i) * do_stride + (int64_t)h * d;
  for (int c = tid; c < d; c += F32_NT) {
    sq_row[c] = qr[c];
    sdo_row[c] = dor[c];
  }
  __syncthreads();
  const float li = lse[((int64_t)b * hq + h) * max_sq + i];
  const float di = delta[((int64_t)b * hq + h) * max_sq + i];
  const int kend = causal ? (i + 1 < sk ? i + 1 : sk) : sk;
  float acc[F32_MAXC] = {0.f, 0.f};
  for (int j0 = 0; j0 < kend; j0 += F32_NT) {
    const int j = j0 + tid;
    float ds = 0.f;
    if (j < kend) {
      const float s = scale * dot_row(sq_row, k + (int64_t)(k0 + j) * k_stride + (int64_t)hkv * d, d);
      const float pj = expf(s - li);
      const float dp = dot_row(sdo_row, v + (int64_t)(k0 + j) * v_stride + (int64_t)hkv * d, d);
      ds = pj * (dp - di);
    }
    sds[tid] = ds;
    __syncthreads();
    const int cnt = kend - j0 < F32_NT ? kend - j0 : F32_NT;
#pragma unroll
    for (int ci = 0; ci < F32_MAXC; ++ci) {
      const int c = tid + ci * F32_NT;
      if (c < d) {
        float a = acc[ci];
        const float *kp = k + (int64_t)(k0 + j0) * k_stride + (int64_t)hkv * d + c;
        for (int jj = 0; jj < cnt; ++jj) a += sds[jj] * kp[(int64_t)jj * k_stride];
        acc[ci] = a;
      }
    }
    __syncthreads();
  }
  float *dqr = dq + (int64_t)(q0 + i) * dq_stride + (int64_t)h * d;
#pragma unroll
  for (int ci = 0; ci < F32_MAXC; ++ci) {
    const int c = tid + ci * F32_NT;
    if (c < d) dqr[c] = accumulate ? dqr[c] + acc[ci] * scale : acc[ci] * scale;
  }
}

// dK, dV: one block per key/value row; walks the query heads of its group and the
// query rows that attend to it.
__global__ void __launch_bounds__(F32_NT)
attn_bwd_dkv_f32_kernel(const float *__restrict__ dout, const float *__restrict__ q, const float *__restrict__ k,
                        const float *__restrict__ v, const float *__restrict__ lse,
                        const float *__restrict__ delta, float *__restrict__ dk, float *__restrict__ dv,
                        const int32_t *__restrict__ cu_q, const int32_t *__restrict__ cu_k, int max_sq, int hq,
                        int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t do_stride,
                        int64_t dk_stride, int64_t dv_stride, float scale, int causal) {
  __shared__ float sk_row[256], sv_row[256];
  __shared__ float sp[F32_NT], sds[F32_NT];
  const int b = blockIdx.z, hkv = blockIdx.y, j = blockIdx.x;
  const int q0 = cu_q[b], sq = cu_q[b + 1] - q0;
  const int k0 = cu_k[b], sk = cu_k[b + 1] - k0;
  if (j >= sk) return;
  const int tid = threadIdx.x;
  const int ratio = hq / hk;
  const float *kr = k + (int64_t)(k0 + j) * k_stride + (int64_t)hkv * d;
  const float *vr = v + (int64_t)(k0 + j) * v_stride + (int64_t)hkv * d;
  for (int c = tid; c < d; c += F32_NT) {
    sk_row[c] = kr[c];
    sv_row[c] = vr[c];
  }
  __syncthreads();
  const int ibeg = causal ? j : 0;
  float ak[F32_MAXC] = {0.f, 0.f}, av[F32_MAXC] = {0.f, 0.f};
  for (int g = 0; g < ratio; ++g) {
    const int h = hkv * ratio + g;
    for (int i0 = ibeg; i0 < sq; i0 += F32_NT) {
      const int i = i0 + tid;
      float pj = 0.f, ds = 0.f;
      if (i < sq) {
        const float s = scale * dot_row(sk_row, q + (int64_t)(q0 + i) * q_stride + (int64_t)h * d, d);
        pj = expf(s - lse[((int64_t)b * hq + h) * max_sq + i]);
        const float dp = dot_row(sv_row, dout + (int64_t)(q0 + i) * do_stride + (int64_t)h * d, d);
        ds = pj * (dp - delta[((int64_t)b * hq + h) * max_sq + i]);
      }
      sp[tid] = pj;
      sds[tid] = ds;
      __syncthreads();
      const int cnt = sq - i0 < F32_NT ? sq - i0 : F32_NT;
#pragma unroll
      for (int ci = 0; ci < F32_MAXC; ++ci) {
        const int c = tid + ci * F32_NT;
        if (c < d) {
          float a1 = ak[ci], a2 = av[ci];
          const float *qp = q + (int64_t)(q0 + i0) * q_stride + (int64_t)h * d + c;
          const float *dp_ = dout + (int64_t)(q0 + i0) * do_stride + (int64_t)h * d + c;
          for (int ii = 0; ii < cnt; ++ii) {
            a1 += sds[ii] * qp[(int64_t)ii * q_stride];
            a2 += sp[ii] * dp_[(int64_t)ii * do_stride];
          }
          ak[ci] = a1;
          av[ci] = a2;
        }
      }
      __syncthreads();
    }
  }
  float *dkr = dk + (int64_t)(k0 + j) * dk_stride + (int64_t)hkv * d;
  float *dvr = dv + (int64_t)(k0 + j) * dv_stride + (int64_t)hkv * d;
#pragma unroll
  for (int ci = 0; ci < F32_MAXC; ++ci) {
    const int c = tid + ci * F32_NT;
    if (c < d) {
      dkr[c] = ak[ci] * scale;
      dvr[c] = av[ci];
    }
  }
}

int attn_fwd_f32(const void *q, const void *k, const void *v, void *out, float *lse, const int32_t *cu_q,
                 const int32_t *cu_k, int batch, int max_sq, int max_sk, int hq, int hk, int d, int64_t q_stride,
                 int64_t k_stride, int64_t v_stride, int64_t o_stride, float scale, int causal, hipStream_t st) {
  DH_CHECK(q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 && aligned16(q) && aligned16(k) && aligned16(v),
           "fp32 attention needs 16-byte aligned rows");
  if (d <= 128) {
    return (d == 64 ? attn_fwd_f32_mma<64, true> : d < 64 ? attn_fwd_f32_mma<64, false>
            : d == 128 ? attn_fwd_f32_mma<128, true> : attn_fwd_f32_mma<128, false>)(
        (const float *)q, (const float *)k, (const float *)v, (float *)out, lse, cu_q, cu_k, batch, max_sq, hq, hk, d, q_stride,
        k_stride, v_stride, o_stride, scale, causal, st);
  }
  hipLaunchKernelGGL(attn_fwd_f32_kernel, dim3((unsigned)max_sq, (unsigned)hq, (unsigned)batch), dim3(F32_NT), 0, st,
                     (const float *)q, (const float *)k, (const float *)v, (float *)out, lse, cu_q, cu_k, max_sq, hq,
                     hk, d, q_stride, k_stride, v_stride, o_stride, scale, causal);
  DH_LAUNCH_CHECK();
  return DH_OK;
}

int attn_bwd_f32(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                 void *dq, void *dk, void *dv, const int32_t *cu_q, const int32_t *cu_k, int batch, int max_sq,
                 int max_sk, int hq, int hk, int d, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                 int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride, float scale, int causal,
                 int dq_accumulate, hipStream_t st) {
  DH_CHECK(q_stride % 4 == 0 && k_stride % 4 == 0 && v_stride % 4 == 0 && do_stride % 4 == 0 && aligned16(q) &&
               aligned16(k) && aligned16(v) && aligned16(dout),
           "fp32 attention needs 16-byte aligned rows");
  if (d <= 128) {
    return (d == 64 ? attn_bwd_f32_mma<64, true> : d < 64 ? attn_bwd_f32_mma<64, false>
            : d == 128 ? attn_bwd_f32_mma<128, true> : attn_bwd_f32_mma<128, false>)(
        (const float *)dout, (const float *)q, (const float *)k, (const float *)v, lse, delta, (float *)dq, (float *)dk,
        (float *)dv, cu_q, cu_k, batch, max_sq, max_sk, hq, hk, d, q_stride, k_stride, v_stride, do_stride, dq_stride,
        dk_stride, dv_stride, scale, causal, dq_accumulate, st);
  }
  if (max_sq > 0)
    hipLaunchKernelGGL(attn_bwd_dq_f32_kernel, dim3((unsigned)max_sq, (unsigned)hq, (unsigned)batch), dim3(F32_NT), 0,
                       st, (const float *)dout, (const float *)q, (const float *)k, (const float *)v, lse, delta,
                       (float *)dq, cu_q, cu_k, max_sq, hq, hk, d, q_stride, k_stride, v_stride, do_stride, dq_stride,
                       scale, causal, dq_accumulate);
  if (max_sk > 0)
    hipLaunchKernelGGL(attn_bwd_dkv_f32_kernel, dim3((unsigned)max_sk, (unsigned)hk, (unsigned)batch), dim3(F32_NT),
                       0, st, (const float *)dout, (const float *)q, (const float *)k, (const float *)v, lse, delta,
                       (float *)dk, (float *)dv, cu_q, cu_k, max_sq, hq, hk, d, q_stride, k_stride, v_stride,
                       do_stride, dk_stride, dv_stride, scale, causal);
  DH_LAUNCH_CHECK();
  return DH_OK;
}

}  // namespace dh
