// Device pieces shared by the tiled GEMM families (gemm_tile.hip,
// gemm_split.hip): tile order, and how a 16-bit operand of either storage
// order is staged in LDS and read back as MFMA 16x16x32 fragments.
#pragma once

#include "common.h"

namespace mk {

typedef short ts16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) ts16x4* lds_ts16x4_ptr;

// XOR of the 32-byte piece index of k row k in a staged [k][BX] operand.  A
// transposing read takes 32 bytes of rows 8g + r (r = 0..3; g = 0, 1 in one
// half wave, 2, 3 in the other): rows of BX * 2 bytes wrap 256 bytes of
// banks after 128 / BX rows, so the bits of k that do not move the bank by
// themselves move the piece.
template <int BX>
__device__ __forceinline__ int swz_x(int k) {
  if constexpr (BX >= 128) return (k & 3) | (((k >> 3) & 1) << 2);
  else if constexpr (BX == 64) return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
  else if constexpr (BX == 32) return (k >> 3) & 1;
  else return 0;
}

// Logical workgroup id that keeps runs of consecutive ids on one XCD, for
// any grid size (workgroup b runs on XCD b % 8).
__device__ __forceinline__ int xcd_run_id(int b, int n) {
  const int x = b & 7, q = n >> 3, r = n & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// One operand's staging coordinates: 1 KB piece q of a step (64 lanes x 16
// bytes) -> this lane's tile row / first tile column x and its k.
template <int BX, bool XC>  // XC: x contiguous in memory
__device__ __forceinline__ void stage_coord(int q, int lane, int& x, int& k) {
  if constexpr (XC) {
    constexpr int CPR = BX / 8;  // 16-byte chunks per k row
    k = q * (64 / CPR) + lane / CPR;
    x = 8 * ((lane % CPR) ^ (2 * swz_x<BX>(k)));
  } else {
    constexpr int PS = BX / 16;  // pieces per 32 k
    x = 16 * (q % PS) + (lane >> 2);
    k = 32 * (q / PS) + 8 * ((lane & 3) ^ ((x >> 1) & 3));
  }
}

// Byte offset, within an operand's step, of this lane's fragment piece of
// the 16-wide tile at w0 (k 0..31; + 1024 per 16 rows and + 64 BX per 32 k
// when k is contiguous, + 64 BX per 32 k otherwise).
template <int BX, bool XC>
__device__ __forceinline__ int frag_offset(int w0, int lane) {
  if constexpr (XC) {
    const int g = lane >> 4, r = (lane & 15) >> 2, q = lane & 3;
    const int k = 8 * g + r, col = w0 + 4 * q;
    return k * (BX * 2) + 16 * ((col >> 3) ^ (2 * swz_x<BX>(k))) + 2 * (col & 7);
  } else {
    const int row = w0 + (lane & 15);
    return row * 64 + 16 * ((lane >> 4) ^ ((row >> 1) & 3));
  }
}

template <int BX, bool XC>
__device__ __forceinline__ u32x4 read_frag(const unsigned char* p) {
  if constexpr (XC) {
    const ts16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ts16x4_ptr)(p));
    const ts16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ts16x4_ptr)(p + 8 * BX));
    const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
    return u32x4{l.x, l.y, h.x, h.y};
  } else {
    return *reinterpret_cast<const u32x4*>(p);
  }
}

// This workgroup's tile: bands of 4 tile rows, consecutive ids down a band's
// columns, so the panels that neighbours share stay in one XCD's L2.
__device__ __forceinline__ void tile_origin(int M, int N, int bm, int bn, int& m0, int& n0) {
  const int tiles_m = (M + bm - 1) / bm, tiles_n = (N + bn - 1) / bn;
  const int L = xcd_run_id(blockIdx.x, gridDim.x);
  const int band = L / (4 * tiles_n), left = tiles_m - 4 * band, h = left < 4 ? left : 4;
  const int r = L - band * 4 * tiles_n;
  m0 = (4 * band + r % h) * bm;
  n0 = (r / h) * bn;
}

}  // namespace mk
