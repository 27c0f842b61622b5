// Dense block-FP8 linear (several rows): argument block and launcher.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace glm53 {

struct DenseArgs {
  const uint8_t* a_hi;     // [rows, K] split activations
  const uint8_t* a_lo;
  const float* a_scale;    // [rows, K / 128]
  const uint8_t* weight;   // [N, K], 16-byte aligned
  const float* scale;      // [ceil(N / 128), K / 128]
  const int32_t* flag;     // device flag of 0x7F / 0xFF weight codes, or null: the kernel looks for them
  int64_t rows, K, N;      // K % 128 == 0, N % 16 == 0
  uint16_t* out;           // [rows, N] bf16
};

// Rows x columns of the output that one workgroup computes.
struct DenseTile {
  int rows, cols;
};
// The tile for a [rows, K] x [N, K] product: up to 32 x 64 run by
// launch_dense_linear, larger ones by the grouped GEMM (tile_rows = rows;
// 128 rows: launch_wide_dense with cols / 128 weight tiles per wavefront).
DenseTile dense_tile(int64_t rows, int64_t K, int64_t N);
hipError_t launch_dense_linear(const DenseArgs& a, DenseTile tile, hipStream_t st);

}  // namespace glm53
