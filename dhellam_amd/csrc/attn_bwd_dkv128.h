// dK/dV at head dim 128 in 16 bits: one wavefront on a SIMD, every instruction of the main loop in a fixed order.
#pragma once
#include "attn_loops.inc"
#include "attn_rows.h"

#include <type_traits>

namespace dh {

// A workgroup of four wavefronts owns 64 key rows; each wavefront holds all of them (dK and dV: 256 accumulator registers, V: 64
// registers, K in LDS) and takes every fourth tile of 32 query rows of every head of its group.  The tiles are the wavefront's own: it
// copies the next one to LDS (two stages) while it works on the current one, and no barrier stands in the loop.
// A tile is 128 MFMAs in four phases of 32, and the vector work lies beneath those that do not need it:
//   S = Q K^T   | dP = dO V^T - delta | dV^T += dO^T P   | dK^T += Q^T dS
//   copies      | P = 2^(S c - lse)   | rest of P, dS    | scalar work, first reads of the next tile
// The key index is on lanes in S and dP, so P and dS are operands of the last two as they are; -delta is what dP's
// accumulators start from.  A query or dO fragment serves four MFMAs (64 keys), so that LDS is read at half the rate of two
// wavefronts a SIMD with 32 keys each (68 reads of 16 and 8 bytes a lane for 128 MFMAs), and P and dS cost 128 vector
// instructions a tile.  The loop is written by attn_loops.py.
// What it measured: 2510 cycles a tile, of which the matrix pipe is busy 2048; the kernel of eight wavefronts before it took
// 5300 for the same work, this loop left to the compiler with its instructions in the same order 3300 (an s_nop behind each
// instruction of assembly, no reads across the tile's end).  16x16x32 MFMAs rather than 32x32x16 because the board is bound by power:
// left to the compiler the loop took 3020 cycles with 32x32x16 and 3300 with 16x16x32, but 245 us (1.63 GHz) and 228 (1.9 GHz).
// dK/dV of 32 query / 8 kv heads, 4096 rows x 2048 keys 300 -> 211 us (1.30 PFLOP/s at 1.5 GHz), causal 4096 304 -> 213, 8 / 1 heads x
// 4096 keeping dS 95 -> 77, seven packed sequences of 1 to 3324 tokens 444 -> 300.
// Rows past the sequence are zeros in LDS (buffer descriptors) and in the lse / delta planes: P = 1 there meets dO = 0, and dS = 0.
// Where a key may have no other row (the diagonal's tiles) they are masked: the score of a row of zeros and a key that holds an
// infinity is none.  Key blocks that no row of a tile sees get no products: a row's dO that is not finite reaches dV and dK of the
// keys in its block of 32 and before, no further.
// The wavefronts' partial sums go through LDS and are added in the order of the wavefronts.
template <typename T, bool STORE_DS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) attn_bwd_dkv128_kernel(const AttnBwdParams p) {
  constexpr int D = 128, BN = 64, BM = 32, NW = 4;
  constexpr uint32_t ROWB = 2 * D, QTB = BM * ROWB;                  // bytes of a row and of a Q (or dO) tile
  constexpr uint32_t LD = 2 * QTB, SLOTB = 2 * QTB + 256;            // lse and -delta behind the two tiles
  constexpr uint32_t WAVEB = 2 * SLOTB, KT = NW * WAVEB;             // two stages a wavefront; the K tile
  constexpr uint32_t LDS_BYTES = KT + BN * ROWB;
  static_assert(LDS_BYTES >= NW * 8 * 4096, "exchange area");
  __shared__ __attribute__((aligned(1024))) char sAll[LDS_BYTES];

  const int b = __builtin_amdgcn_readfirstlane(seq_by_length(p.cu_q, gridDim.y, blockIdx.y));
  const int G = p.hk * p.hsplit;
  int hg, px;
  xcd_group_item(blockIdx.x, G, gridDim.x / G, hg, px);
  const int hkv = hg / p.hsplit, hs = hg % p.hsplit;
  const int q0 = p.cu_q[b] >> p.q_shift, sq = (p.cu_q[b + 1] >> p.q_shift) - q0;
  const int k0 = p.cu_k[b] >> p.k_shift, sk = (p.cu_k[b + 1] >> p.k_shift) - k0;
  const int nkt = (sk + BN - 1) / BN;
  const int causal = p.causal;
  int kt0 = px, kt1 = 0, nk = 1;
  if (causal) {                                       // key tiles j and n - 1 - j: every workgroup does the same amount of work
    if (2 * px >= nkt) return;
    kt1 = nkt - 1 - px;                               // (the one of the early keys has more rows: first)
    nk = kt0 == kt1 ? 1 : 2;
  } else if (px >= nkt) {
    return;
  }
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hper = p.hq / p.hk / p.hsplit;
  const int h_first = hkv * (p.hq / p.hk) + hs * hper;
  const uint32_t lds0 = (uint32_t)(uintptr_t)sAll;
  const uint32_t wbase = lds0 + (uint32_t)w * WAVEB;

  const uint32_t q_rowb = (uint32_t)p.q_stride * 2u, do_rowb = (uint32_t)p.do_stride * 2u, k_rowb = (uint32_t)p.k_stride * 2u;

  for (int ki = 0; ki < nk; ++ki) {
    const int j0 = (ki == 0 ? kt0 : kt1) * BN;
    // lane addresses, formed anew for each key tile: nothing but the lane id lives through the sums at its end
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int r = lane & 15, g = lane >> 4;
    uint32_t cq[4], cd[4], ck[4];
    rows_lanes(cq, lane, q_rowb);
    rows_lanes(cd, lane, do_rowb);
    rows_lanes(ck, lane, k_rowb);
    const uint32_t c_ld = (uint32_t)(lane & 31) * 4u + (lane >> 5 ? (uint32_t)(p.ld2_plane * 4) : 0u);
    // fragment reads: row r, chunk 4 ks + g; transposed: rows 4 g + r / 4 (and 16 further), chunk 2 t + (r % 4) / 2
    uint32_t rq[4], rk[4], ta[8];
    {
      const uint32_t row = (uint32_t)(r * ROWB), x = (uint32_t)((g ^ swz16(r)) << 4);
#pragma unroll
      for (uint32_t ks = 0; ks < 4; ++ks) {
        rq[ks] = wbase + row + (x ^ (ks << 6));
        rk[ks] = lds0 + KT + row + (x ^ (ks << 6));
      }
      const int tr = 4 * g + (r >> 2), ch = (r & 3) >> 1;
      const uint32_t at = wbase + (uint32_t)(tr * ROWB + 8 * (r & 1));
#pragma unroll
      for (int t = 0; t < 8; ++t) ta[t] = at + (uint32_t)(((ch ^ swz16(tr)) ^ (2 * t)) << 4);
    }
    const uint32_t ldr = wbase + LD + 16 * (uint32_t)g;

    // K and V tile: 16 rows of each a wavefront (zeros past the end; those columns of dK and dV are not stored).  V waits in the
    // second stages for being read as fragments: gathered from memory, 16 rows of 64 bytes a load in every wavefront, it cost 1 % of a long
    // backward and 3 % of a batch of short ones (whole calls, seven documents 710 -> 705 us, 16 heads, eight sequences of 12 to 748 rows 92 -> 90).
    {
      const int row = j0 + 16 * w, rows = sk - row < 16 ? sk - row : 16;
      const uint32_t v_rowb = (uint32_t)p.v_stride * 2u;
      const int4v rsk = rows_rsrc(reinterpret_cast<const T *>(p.k) + (int64_t)(k0 + row) * p.k_stride + (int64_t)hkv * D,
                                  rows > 0 ? (uint32_t)(rows - 1) * k_rowb + ROWB : 0u);
      const int4v rsv = rows_rsrc(reinterpret_cast<const T *>(p.v) + (int64_t)(k0 + row) * p.v_stride + (int64_t)hkv * D,
                                  rows > 0 ? (uint32_t)(rows - 1) * v_rowb + ROWB : 0u);
      uint32_t cv[4];
      rows_lanes(cv, lane, v_rowb);
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x) {
        copy_1k(cv[x], rsv, 0u, wbase + SLOTB + 1024u * x);
        copy_1k(ck[x], rsk, 0u, lds0 + KT + (uint32_t)w * 16 * ROWB + 1024u * x);
      }
    }
    const int i_begin = causal ? j0 : 0;
    const int ntq = i_begin < sq ? (sq - i_begin + BM - 1) / BM : 0;
    const int total = ntq * hper;

    // the wavefront's first tile, and how the loop goes on from it: four tiles further, or to the same place of the next head
    int rem = total > w ? (total - w + NW - 1) / NW : 0, ct = w, ch = h_first;
    while (rem > 0 && ct >= ntq) { ct -= ntq; ++ch; }
    const int64_t row = (int64_t)q0 + i_begin + ct * BM;
    const T *qp = reinterpret_cast<const T *>(p.q) + row * p.q_stride + (int64_t)ch * D;
    const T *dp = reinterpret_cast<const T *>(p.dout) + row * p.do_stride + (int64_t)ch * D;
    const float *lp = p.ld2 + ((int64_t)b * p.hq + ch) * p.ld2_pitch + (i_begin + ct * BM);
    const int64_t qstep = (int64_t)NW * BM * q_rowb, dstep = (int64_t)NW * BM * do_rowb;
    const int64_t qwrap = (int64_t)ROWB - (int64_t)ntq * BM * q_rowb, dwrap = (int64_t)ROWB - (int64_t)ntq * BM * do_rowb;
    const int64_t lwrap = ((int64_t)p.ld2_pitch - (int64_t)ntq * BM) * 4;
    const uint32_t ldbytes = (uint32_t)(p.ld2_plane * 4) + 128u, q16 = 16u * q_rowb, d16 = 16u * do_rowb;
    // tiles with scores to mask: the first two of a causal one; and which of them the rows end in
    const int rows = sq - i_begin, mct = causal ? 2 : 0, pct = (rows & (BM - 1)) != 0 ? ntq - 1 : -1;
    {
      const int left = rows - ct * BM < BM ? rows - ct * BM : BM;
      const int4v rsq = rows_rsrc(qp, rem > 0 ? (uint32_t)(left - 1) * q_rowb + ROWB : 0u);
      const int4v rsd = rows_rsrc(dp, rem > 0 ? (uint32_t)(left - 1) * do_rowb + ROWB : 0u);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        copy_1k(cq[i & 3], rsq, i < 4 ? 0u : q16, wbase + 1024u * i);
        copy_1k(cd[i & 3], rsd, i < 4 ? 0u : d16, wbase + QTB + 1024u * i);
      }
      copy_256(c_ld, rows_rsrc(lp, rem > 0 ? ldbytes : 0u), wbase + LD);
    }
    int4v V[4][4];
    {
      typedef __attribute__((address_space(3))) const int4v *lds_i4;
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) V[kb][ks] = *(lds_i4)(rk[ks] - KT + (uint32_t)kb * WAVEB + SLOTB);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // (the loop copies to the second stages)
    }
    const int vx = causal ? r - 4 * g : -(1 << 20);   // key - row of a score, but for what the loop adds
    const int vz = 4 * g - rows;                      // row - rows
    floatx4 dV[4][8], dK[4][8];                       // key block, d block
#define DH_ACC4(x, X, kb, t) [x##kb##t] "=a"(X[kb][t])
#define DH_ACC(x, X, kb)                                                                                                             \
  DH_ACC4(x, X, kb, 0), DH_ACC4(x, X, kb, 1), DH_ACC4(x, X, kb, 2), DH_ACC4(x, X, kb, 3), DH_ACC4(x, X, kb, 4), DH_ACC4(x, X, kb, 5), \
      DH_ACC4(x, X, kb, 6), DH_ACC4(x, X, kb, 7)
#define DH_V4(kb) [V##kb##0] "v"(V[kb][0]), [V##kb##1] "v"(V[kb][1]), [V##kb##2] "v"(V[kb][2]), [V##kb##3] "v"(V[kb][3])
#define DH_LOOP(TEXT, ...)                                                                                                           \
  asm volatile(TEXT                                                                                                                 \
               : DH_ACC(dv, dV, 0), DH_ACC(dv, dV, 1), DH_ACC(dv, dV, 2), DH_ACC(dv, dV, 3), DH_ACC(dk, dK, 0), DH_ACC(dk, dK, 1),      \
                 DH_ACC(dk, dK, 2), DH_ACC(dk, dK, 3), [ct] "+s"(ct), [rem] "+s"(rem)                    \
               : DH_V4(0), DH_V4(1), DH_V4(2), DH_V4(3), [rq0] "v"(rq[0]), [rq1] "v"(rq[1]), [rq2] "v"(rq[2]), [rq3] "v"(rq[3]),       \
                 [rk0] "v"(rk[0]), [rk1] "v"(rk[1]), [rk2] "v"(rk[2]), [rk3] "v"(rk[3]), [ta0] "v"(ta[0]), [ta1] "v"(ta[1]),          \
                 [ta2] "v"(ta[2]), [ta3] "v"(ta[3]), [ta4] "v"(ta[4]), [ta5] "v"(ta[5]), [ta6] "v"(ta[6]), [ta7] "v"(ta[7]),          \
                 [cq0] "v"(cq[0]), [cq1] "v"(cq[1]), [cq2] "v"(cq[2]), [cq3] "v"(cq[3]), [cd0] "v"(cd[0]), [cd1] "v"(cd[1]),          \
                 [cd2] "v"(cd[2]), [cd3] "v"(cd[3]), [cld] "v"(c_ld), [ldr] "v"(ldr), [vx] "v"(vx), [vz] "v"(vz), [scale] "s"(p.scale_log2), \
                 [wbase] "s"(wbase), [ntq] "s"(ntq), [rows] "s"(rows), [mct] "s"(mct), [pct] "s"(pct), [qrowb] "s"(q_rowb), [drowb] "s"(do_rowb),     \
                 [q16] "s"(q16), [d16] "s"(d16), [ldbytes] "s"(ldbytes), [qp] "s"(qp), [dp] "s"(dp), [lp] "s"(lp),                    \
                 [qstep] "s"(qstep), [dstep] "s"(dstep), [qwrap] "s"(qwrap), [dwrap] "s"(dwrap), [lwrap] "s"(lwrap) __VA_ARGS__       \
               : DH_DKV128_CLOBBERS)
    if constexpr (STORE_DS) {
      // packed dS goes out in the order that the dQ product reads: 8 bytes a row block and key block
      const int64_t tile_ds = (int64_t)p.ds_nkb * 2048;
      const char *dsp = reinterpret_cast<const char *>(p.ds) + (((int64_t)b * p.hq + ch) * p.ds_nqt + ((i_begin >> 5) + ct)) * tile_ds + (int64_t)(j0 >> 5) * 2048;
      const int64_t dsstep = NW * tile_ds, dswrap = (int64_t)(p.ds_nqt - ntq) * tile_ds;
      const int dsmask = __builtin_amdgcn_readfirstlane(j0 + BN > sk);
      const int vy = j0 + r - sk;
      const uint32_t dso = (uint32_t)((g & 1) * 512 + r * 16 + (g >> 1) * 8);
      if constexpr (__is_same(T, bf16_t)) DH_LOOP(DH_DKV128_LOOP_BF16_DS, , [dsp] "s"(dsp), [dsstep] "s"(dsstep), [dswrap] "s"(dswrap), [dsmask] "s"(dsmask), [vy] "v"(vy), [dso] "v"(dso));
      else DH_LOOP(DH_DKV128_LOOP_F16_DS, , [dsp] "s"(dsp), [dsstep] "s"(dsstep), [dswrap] "s"(dswrap), [dsmask] "s"(dsmask), [vy] "v"(vy), [dso] "v"(dso));
    } else {
      if constexpr (__is_same(T, bf16_t)) DH_LOOP(DH_DKV128_LOOP_BF16, );
      else DH_LOOP(DH_DKV128_LOOP_F16, );
    }
#undef DH_LOOP
#undef DH_V4
#undef DH_ACC
#undef DH_ACC4
    __syncthreads();                                  // everyone is done with the tiles

    // add the wavefronts' partial sums in their order: wavefront w ends up with key block w.  (Those without a tile have none: of
    // 512 KB through LDS a key tile, 128 are left where sequences are one tile long.)
    const int nact = total < NW ? (total > 1 ? total : 1) : NW;
    typedef __attribute__((address_space(3))) floatx4 *lds_f4;
    auto sum_up = [&](const floatx4 (&acc)[4][8], floatx4 (&sum)[8]) {
      const lds_f4 dst = (lds_f4)(lds0 + (uint32_t)w * 32768u) + lane;
      if (w < nact) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int t = 0; t < 8; ++t) dst[64 * (8 * kb + t)] = acc[kb][t];
      }
      __syncthreads();
      auto add = [&](auto parts) {
#pragma unroll
        for (int x = 0; x < decltype(parts)::value; ++x) {
          const lds_f4 src = (lds_f4)(lds0 + (uint32_t)x * 32768u + (uint32_t)w * 8192u) + lane;
#pragma unroll
          for (int t = 0; t < 8; ++t) sum[t] = x == 0 ? src[64 * t] : sum[t] + src[64 * t];
        }
      };
      if (nact == NW) add(std::integral_constant<int, NW>());
      else if (nact == 3) add(std::integral_constant<int, 3>());
      else if (nact == 2) add(std::integral_constant<int, 2>());
      else add(std::integral_constant<int, 1>());
      __syncthreads();
    };
    floatx4 sK[8], sV[8];
    sum_up(dV, sV);
    sum_up(dK, sK);
    const int jrow = j0 + 16 * w + r;
    if (jrow < sk) {
      if (p.hsplit == 1) {
        struct alignas(8) Four { T v[4]; };
        T *dkp = reinterpret_cast<T *>(p.dk) + (int64_t)(k0 + jrow) * p.dk_stride + (int64_t)hkv * D + 4 * g;
        T *dvp = reinterpret_cast<T *>(p.dv) + (int64_t)(k0 + jrow) * p.dv_stride + (int64_t)hkv * D + 4 * g;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          Four a, bq;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            a.v[e] = static_cast<T>(sK[t][e] * p.scale);
            bq.v[e] = static_cast<T>(sV[t][e]);
          }
          *reinterpret_cast<Four *>(dkp + 16 * t) = a;
          *reinterpret_cast<Four *>(dvp + 16 * t) = bq;
        }
      } else {
        const int64_t off = (((int64_t)hs * p.total_k + (k0 + jrow)) * p.hk + hkv) * D + 4 * g;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          *reinterpret_cast<floatx4 *>(p.dk_part + off + 16 * t) = sK[t] * p.scale;
          *reinterpret_cast<floatx4 *>(p.dv_part + off + 16 * t) = sV[t];
        }
      }
    }
  }
}

}  // namespace dh
