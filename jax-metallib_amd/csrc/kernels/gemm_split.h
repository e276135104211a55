// Host entry of the f32 GEMM (gemm_split.hip): operands of any size, either
// storage order, any row stride.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mkg {

// C[b] = A[b] @ B[b], f32, C row-major [batch, M, N], packed; A and B as in
// TileGemm (gemm_tile.h).
struct SplitGemm {
  const float* a = nullptr;
  const float* b = nullptr;
  float* c = nullptr;
  int64_t batch = 1, M = 0, N = 0, K = 0;
  int64_t lda = 0, ldb = 0, sa = 0, sb = 0;
  bool a_t = false, b_t = false;
};

// tile: 0 the built-in choice, else 16, 64 or 128 rows.  Same bits.
hipError_t split_launch(const SplitGemm& g, int tile, hipStream_t st);

}  // namespace mkg
