// Which products the general dot_general (dot_general.hip) runs on the tiled
// kernels; the planner asks before it leaves an operand where it lies.
#pragma once

#include <stdint.h>

namespace mkg {

// How the tiled kernels read a product's operands in place (TileGemm,
// gemm_tile.h).
struct DotOrder {
  bool a_t = false, b_t = false;
  int64_t lda = 0, ldb = 0;
};

// Whether a floating product runs on them: both operands have one contiguous
// dimension and rows that do not overlap, the sum is long enough, the grid
// fits a launch.  Strides in elements: a (batch, m, k), b (batch, k, n).
bool dot_tiled(int64_t batch, int64_t M, int64_t N, int64_t K, const int64_t* a_strides, const int64_t* b_strides,
               DotOrder* order);

}  // namespace mkg
