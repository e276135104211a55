// Host entry of the tiled 16-bit GEMM family (gemm_tile.hip): bf16 / f16
// products of any size, operands in either storage order with any row
// stride.  Used by the bf16 GEMM C-ABI (gemm.hip) for the shapes its 256-wide
// kernels do not fill or divide, and by the general dot_general
// (dot_general.hip) for transposed, odd-sized and f16 operands.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mkg {

// C[b] = A[b] @ B[b], C row-major [batch, M, N], packed.
//   A[m, k] at a + b*sa + m*lda + k   (a_t: at b*sa + k*lda + m)
//   B[k, n] at b + b*sb + k*ldb + n   (b_t: at b*sb + n*ldb + k)
// in elements; every element in that index range must be readable.
struct TileGemm {
  const void* a = nullptr;
  const void* b = nullptr;
  void* c = nullptr;
  const void* aux = nullptr;  // epi: bf16, C's layout (bf16 output, N % 4 == 0)
  int64_t batch = 1, M = 0, N = 0, K = 0;
  int64_t lda = 0, ldb = 0, sa = 0, sb = 0;
  bool a_t = false, b_t = false;
  bool f16 = false;      // operands (and a 16-bit result) f16, else bf16
  bool out_f32 = false;  // f32 result, else the operands' type
  int epi = 0;           // MK_EPI_NONE / MK_EPI_ADD / MK_EPI_SWIGLU
  bool registers = false;  // feed through registers whatever the alignment
};

// Tile shapes, smallest first.
enum TileShape { T16x64 = 0, T32x64, T64x64, T128x64, T128x128, T256x256, kTileShapes };

// Whether an M x N result's tiles of that shape fit a launch (2^32 threads in
// the grid's first dimension), fed either way.
bool tile_grid_fits(int64_t M, int64_t N, int shape);

// Whether the operands' alignment lets LDS DMA feed the tiles (16-byte
// pieces never straddle a row's end); otherwise registers do.
bool tile_dma_ok(const TileGemm& g);

// The shape the family takes for this product (tile_dma_ok included), of those
// whose grid fits.
int tile_pick(const TileGemm& g);

// Estimated microseconds of the product in that shape, launch not counted.
double tile_estimate(const TileGemm& g, int shape);

hipError_t tile_launch(const TileGemm& g, int shape, hipStream_t st);

}  // namespace mkg
