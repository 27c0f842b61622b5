// Dense block-FP8 linear (several rows): argument block and launcher.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace glm53 {

struct DenseArgs {
  const uint16_t* x;       // [rows, K] bf16 activations, 16-byte aligned, or null: a_hi, a_lo, a_scale hold their split
  const uint8_t* a_hi;     // [rows, K]; for launch_dense_linear in MFMA operand order
  const uint8_t* a_lo;
  const float* a_scale;    // [rows, K / 128]
  const uint8_t* weight;   // [N, K], 16-byte aligned
  const float* scale;      // [ceil(N / 128), K / 128]
  const int32_t* flag;     // device flag of 0x7F / 0xFF weight codes, or null: the kernel looks for them
  // gate / up / SwiGLU (launch_dense_linear's swiglu): weight holds the gate
  // rows, weight_up the up rows of the same shape, out = SwiGLU
  const uint8_t* weight_up;
  const float* scale_up;
  const int32_t* flag_up;
  float limit;
  int64_t rows, K, N;      // K % 128 == 0, N % 16 == 0
  uint16_t* out;           // [rows, N] bf16
};

// Rows x output columns that one workgroup computes.
struct DenseTile {
  int rows, cols;
};
// The tile for a [rows, K] x [N, K] product, or (swiglu) for the SwiGLU of
// two of them: up to 32 rows x 64 weight columns run by launch_dense_linear,
// larger ones by the grouped GEMM (tile_rows = rows; 128 rows:
// launch_wide_dense with weight columns / 128 tiles per wavefront).
DenseTile dense_tile(int64_t rows, int64_t K, int64_t N, bool swiglu);
// Whether launch_dense_linear runs the tile.
inline bool dense_ksplit(DenseTile t, bool swiglu) { return t.rows <= 32 && (swiglu ? 2 : 1) * t.cols <= 64; }
// Whether launch_dense_linear takes the tile's bf16 activations as they are
// (DenseArgs.x) and splits them itself.
bool dense_splits_x(DenseTile t, int64_t K, bool swiglu);
hipError_t launch_dense_linear(const DenseArgs& a, DenseTile tile, bool swiglu, hipStream_t st);

}  // namespace glm53
