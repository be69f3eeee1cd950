// Dense products of fp32 matrices on fp32 MFMAs.
#pragma once
#include <cstdint>

namespace dh {

// D [rows, cols] (+)= X Y: X is [rows, k], or [k, rows] where x_strided; Y is [cols, k] (its transpose), or [k, cols] where y_strided.
// All dense.
struct GemmF32 {
  const float *x, *y;
  float *d;
  int64_t rows, cols, k;
  bool x_strided, y_strided, accumulate;
};

// Whether launch_gemm_f32 takes the product and is the faster one.
bool gemm_f32_pays(const GemmF32 &g);
int launch_gemm_f32(const GemmF32 &g, void *stream);

}  // namespace dh
