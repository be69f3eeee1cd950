// Which of the families of 16-bit attention kernels a call at head dim 128 takes: the hand-ordered ones, one workgroup a compute unit and
// causal ones all of one length (dK/dV always, the forward and the recomputing dQ where tiles of 256 or 128 rows pay, on one wavefront a SIMD: fwd_rows
// and dq_rows; else on two, 512 threads), or the compiler-scheduled ones that run the other head dims (smaller workgroups, shorter start and
// end).  Host code, shared by forward and backward.
#pragma once
#include <float.h>
#include <stdint.h>

namespace dh {

// The scale of scores in exp2 units.  Masked scores are -inf ahead of the scale, so that 0 times them would be none: the smallest normal
// number takes its place, which leaves finite scores where 0 puts them.
static inline float attn_scale_log2(float scale) { return scale == 0.f ? FLT_MIN : scale * 1.4426950408889634f; }

// Workgroups of a hand-ordered kernel with query tiles of `rows`: one per tile, causal ones take two.
static inline int64_t attn_wgs(int max_sq, int rows, int hq, int batch, int causal) {
  const int64_t t = (max_sq + rows - 1) / rows;
  return (causal ? (t + 1) / 2 : t) * hq * batch;
}

// Calls of several lengths that are not causal, where the kernels of one wavefront a SIMD pay: their tiles start and end in as many cycles as 10
// to 14 tiles of keys take, so the sequences are 350 rows long on average, and 256-row tiles, of which half a one lies past each sequence's end,
// fill 70 % of their rounds of 256 workgroups.  us, whole calls, eight wavefronts / here: 32 heads, 12 sequences of 54 to 782 rows (average 340)
// 344 / 390, 16 x 10 to 448 (129) 99.5 / 104, 16 heads 778 to 2 (268 workgroups by this count, 288 in fact) 155 / 159; but 32 x 84 to
// 624 (352) 236 / 226, 32 x 169 to 755 (446) 324 / 283, 32 / 8 x 300 to 1029 (604) 545 / 464, 16 x 84 to 2620 (1280) 863 / 775.
static inline bool attn_long_rows(int64_t total_q, int batch) { return total_q >= 350ll * batch; }
static inline bool attn_ragged_fills(int hq, int batch, int64_t total_q) {
  const double wgs = ((double)total_q / 256 + 0.5 * batch) * hq;
  return wgs >= 0.7 * 256 * (double)(((int64_t)wgs + 255) / 256);
}

// Largest token stride (elements) of the kernels with one wavefront a SIMD: 32 rows of it are less than 4 GiB, the reach of a copy.
constexpr int64_t ROWS_MAX_STRIDE = 1ll << 26;

// fewest workgroups of 128 query rows for which the 128-row kernels are taken
constexpr int ATTN_128ROW_MIN_WG = 256;

// Causal calls: whether the hand-ordered forward / recomputing dQ kernel is the faster one.  Its workgroups run in rounds
// of 256 (compute units), so what counts is how full the last round is; sequences shorter than the longest have fewer of
// them (`total_q` rows altogether: the share of the longest sequence's grid that has work).  Forward, us, eight wavefronts / other:
//   one length, full rounds (85 % of the places): 8 heads x 2 x 2048 34 / 39, 8 x 4 x 2048 50 / 71, 32 x 4 x 4096 624 / 706,
//     16 x 16 x 700 85 / 96; not full: 8 heads x 4 x 3000 111 / 102, 12 x 11264 536 / 444, 32 x 4352 232 / 193;
//   several lengths (the longest first, so that rounds overlap): from two rounds of real work on it does not matter how
//     they come out: 1 to 3324 tokens x 32 heads (4 rounds) 215 / 225; 3000 + 2 x 1000 x 32 (2.5) 129 / 138; with one round only where the
//     longest is long: 4096 + 2000 + 300 x 16 (1.6) 120 / 129, but 4 to 1423 x 32 (1.1) 54 / 48, 1575 + 302 x 32 (1.0) 54 / 43;
//   64-row tiles need long rows as well: 8 heads x 4096 52 / 69, 16 x 2048 35 / 38, but 32 x 1024 26 / 25, 8 x 8 x 512 22 / 18;
//   128-row ones from 512 on: 32 x 4 x 512 28 / 30, but 16 x 32 x 300 86 / 71.
// The dQ pass follows the forward: with eight wavefronts it gained or lost between 1 and 20 % on the same side.  On one wavefront a SIMD it would be the
// faster one beyond the line too (whole backward, other dQ / hand-ordered: 32 x 4352 646 / 640, 12 x 11264 1283 / 1261, 8 x 4 x 3000 305 / 277, 32 x 1575 +
// 302 137 / 121; but 16 x 4096 + 2000 + 300, on this side, 326 / 323).
static inline bool attn_causal_fills(int max_sq, int hq, int batch, int64_t total_q) {
  if (max_sq <= 0 || batch <= 0) return false;
  const bool big = attn_wgs(max_sq, 128, hq, batch, 1) >= ATTN_128ROW_MIN_WG;
  const int64_t bound = (int64_t)batch * max_sq, rows = total_q < bound ? total_q : bound;
  const int64_t real = (int64_t)((double)attn_wgs(max_sq, big ? 128 : 64, hq, batch, 1) * (double)rows / (double)bound);
  if (max_sq < (big ? 512 : 1536) || real < 240) return false;
  if (big && 10 * rows < 9 * bound) return real >= (max_sq >= 2560 ? 256 : 512);
  return 20 * real >= 17 * 256 * ((real + 255) / 256);
}

}  // namespace dh
