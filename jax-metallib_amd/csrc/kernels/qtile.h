// Host entry of the mid-row quantized matmul (qtile.hip), used by the
// dequant-matmul C-ABI (qmatmul.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mkq {

struct QTilePlan {
  int bm;          // tile rows: 32, 64, 96 or 128
  int ks;          // K split
  int64_t bytes;   // workspace: 64 KB of arrival counters, then partials (0 for ks == 1)
  double us;       // estimated time
};

// The launch for the shape, its workspace at most `cap` bytes; false if the
// kernel does not take it (K % 64 == 0, N % 8 == 0, 32-bit offsets).
bool qtile_plan(bool int4, int64_t M, int64_t K, int64_t N, int64_t cap, QTilePlan* p);

// Whether the pointers have the alignment of the kernel's vector accesses.
bool qtile_aligned(bool int4, const void* x, const void* w, const void* s, const void* z, const void* y,
                   const void* aux, int64_t N);

// Operands as for qgemm_launch; workspace per the plan, counters zeroed (and
// left at zero).
hipError_t qtile_launch(bool int4, const void* x, const void* w, const void* s, const void* z, void* y, int64_t M,
                        int64_t K, int64_t N, const void* aux, int epi, const QTilePlan& p, void* workspace,
                        hipStream_t stream);

}  // namespace mkq
