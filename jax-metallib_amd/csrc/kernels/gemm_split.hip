// f32 GEMM for gfx950 on the bf16 matrix cores.
//
// The f32 MFMA (16x16x4) has 1/16 of the bf16 MFMA's rate.  The split into
// bf16 parts is that of Henry, Tang and Heinecke ("Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", 2019):
// every f32 value is the sum of three bf16 values, x = x1 + x2 + x3 (8
// significant bits each, by rounding to nearest and taking the rest), exactly,
// as long as x3 does not underflow.  So a product is nine bf16 products, of which the three
// smallest (x2 y3, x3 y2, x3 y3: at most 2^-24 of it) are below half an ulp of
// f32; the other six, each exact, are summed in f32 by six bf16 MFMAs of 32 k
// where the f32 MFMA needs eight of 4 k, at 3/8 of their time.  The five
// smaller ones have an accumulator of their own.  Error against 64 bits,
// f32 MFMAs / these: normal inputs K = 64 1.4e-7 / 5.0e-8, K = 1024 5.7e-7 /
// 1.9e-7, K = 4096 1.1e-6 / 3.9e-7; uniform 0..1 K = 1024 4.3e-7 / 1.6e-7.
// 2048^3: 170 -> 92-102 us (0.7 us of a step's 1.4-1.6 is the MFMAs at their
// measured 7 ns each, the rest what the barrier and LDS leave exposed; a
// third LDS slot, a second step of loads in flight and splits placed between
// the MFMAs each changed nothing), 4096^3 1183 -> 751, 1024^3 33 -> 27,
// 1000 x 3000 x 1000 86 -> 50.
//
// What the split cannot represent is recomputed by the f32 MFMA in the same
// launch.  Each result decides for itself, from the largest and the smallest
// nonzero magnitude of its row of A and of its column of B, so its bits are
// those of any tile and whatever else the tile holds:
//   * an infinity, a NaN or a value that rounds to a bf16 infinity leaves a
//     non-finite result: recomputed;
//   * what is below 2^-126 may be lost: parts (2^-125 of an operand) and
//     products and sums of parts (2^-123 a term).  Nothing that counts is if
//     the result is at least K 2^-96 times the larger of 1 and the largest
//     magnitudes (all K losses together are below 2^-26 of it), if the row or
//     the column is all zeros, or if their smallest magnitudes are at least
//     2^-100 (all parts are kept) and have a product of at least 2^-96 (a loss
//     is below 2^-27 of its own term).  Else: recomputed.
// The largest magnitudes are kept while the operands are split.  For the
// smallest a tile with a doubtful result reads its operands again (zeros by
// cancellation among whole numbers, say), and only where they leave one does
// it run the f32 MFMAs, for all of the tile, and take the results in doubt.
// 2048^3, us, a kernel of f32 MFMAs only / this: normal, ReLU and softmax-tail
// data, rows of zeros, operands of 1e-14: 166-184 / 91-100; an infinity in
// each tile 166 / 233, subnormal operands in each 166 / 262, that is the split,
// the second look and the second loop one after the other.
//
// Layout: operands go through registers (f32 loads of 4-byte alignment, one
// step ahead of the MFMAs, two for 16-row tiles), are split there and staged
// as three bf16 planes in the order and swizzle of the 16-bit tile family,
// double buffered.  8 waves (128 x 128), two to a SIMD, so that one's
// splitting runs under the other's MFMAs.
#include "common.h"
#include "gemm_split.h"
#include "gemm_tile_dev.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mk {

struct SplitArgs {
  const float* a;
  const float* b;
  float* c;
  int M, N, K;
  int64_t lda, ldb, sa, sb, sc;
};

typedef f32x4 __attribute__((aligned(4))) f32x4_u4;

struct f32x8 {
  f32x4 lo, hi;
};

// Two floats into three packed bf16 pairs.
__device__ __forceinline__ void split2(float x, float y, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
  p1 = pack_bf16x2(x, y);
  const float rx = x - __uint_as_float(p1 << 16), ry = y - __uint_as_float(p1 & 0xffff0000u);
  p2 = pack_bf16x2(rx, ry);
  p3 = pack_bf16x2(rx - __uint_as_float(p2 << 16), ry - __uint_as_float(p2 & 0xffff0000u));
}

constexpr float kWholeParts = 0x1p-100f;  // operands from here on keep all parts
constexpr float kWholeTerms = 0x1p-96f;   // terms from here on keep all that counts
constexpr uint32_t kInfBits = 0x7f800000u;

template <int BM, int BN, int WM, int WN, int KS, bool AT, bool BT>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_split_kernel(SplitArgs p) {
  constexpr int NW = WM * WN, BK = 32 * KS;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int IA = KS * BM / 16, IB = KS * BN / 16;  // 1 KB pieces of a plane's step
  constexpr int DA = IA / NW, DB = IB / NW;
  static_assert(DA * NW == IA && DB * NW == IB, "the waves share the pieces evenly");
  constexpr int APLANE = IA * 1024, BPLANE = IB * 1024, STEP = 3 * (APLANE + BPLANE);
  constexpr bool AX = AT, BX = !BT;  // the operand's m / n is contiguous

  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int M = p.M, N = p.N, K = p.K;
  int m0, n0;
  tile_origin(M, N, BM, BN, m0, n0);
  const float* A = p.a + (int64_t)blockIdx.z * p.sa;
  const float* B = p.b + (int64_t)blockIdx.z * p.sb;

  // A piece is 8 k of one m (n).  Pieces along contiguous k are loaded as 32
  // bytes and laid out as the 16-bit family's; pieces of an m- (n-)contiguous
  // operand are loaded as 8 floats a k row apart, consecutive lanes taking
  // consecutive columns, so that both end up with k contiguous in LDS (its
  // transposing reads take twice the LDS time for half the bytes).
  int64_t aoff[DA], boff[DB];  // source element at step 0
  int ak[DA], bk[DB], ax[DA], bx[DB], aput[DA], bput[DB];
  auto coord = [&](auto xc, auto tile, int q, int& x, int& k, int& put) {
    constexpr int BXT = decltype(tile)::value;
    if constexpr (decltype(xc)::value) {
      x = (64 * q + lane) % BXT;
      k = 8 * ((64 * q + lane) / BXT);
      put = (k / 32) * 64 * BXT + 64 * x + 16 * (((k / 8) & 3) ^ ((x >> 1) & 3));
    } else {
      stage_coord<BXT, false>(q, lane, x, k);
      put = 1024 * q + 16 * lane;
    }
  };
#pragma unroll
  for (int u = 0; u < DA; ++u) {
    coord(std::bool_constant<AX>{}, std::integral_constant<int, BM>{}, DA * wave + u, ax[u], ak[u], aput[u]);
    const int x = min(m0 + ax[u], M - 1);
    aoff[u] = AX ? (int64_t)ak[u] * p.lda + x : (int64_t)x * p.lda + ak[u];
  }
#pragma unroll
  for (int u = 0; u < DB; ++u) {
    coord(std::bool_constant<BX>{}, std::integral_constant<int, BN>{}, DB * wave + u, bx[u], bk[u], bput[u]);
    const int x = min(n0 + bx[u], N - 1);
    boff[u] = BX ? (int64_t)bk[u] * p.ldb + x : (int64_t)x * p.ldb + bk[u];
  }
  const int64_t astep = AX ? (int64_t)BK * p.lda : BK, bstep = BX ? (int64_t)BK * p.ldb : BK;
  const int NS = (K + BK - 1) / BK, whole = K / BK;  // steps; those that end inside K

  uint32_t* big = reinterpret_cast<uint32_t*>(smem + 2 * STEP);  // largest magnitude of the tile's rows, then columns
  uint32_t* small = big + BM + BN;                               // smallest nonzero one, infinity for none
  uint32_t* flag = small + BM + BN;                              // a result in doubt; one of them finite
  for (int i = tid; i < BM + BN; i += NW * 64) {
    big[i] = 0;
    small[i] = kInfBits;
  }
  if (tid < 2) flag[tid] = 0;

  // Piece w (A's, then B's) of step t; inside: t < whole.
  auto load_piece = [&](int t, int w, bool inside) {
    const bool isa = w < DA;
    const int u = isa ? w : 0, v = isa ? 0 : w - DA;
    const float* s = isa ? A + aoff[u] + t * astep : B + boff[v] + t * bstep;
    const int64_t ld = isa ? p.lda : p.ldb;
    const int kl = K - t * BK - (isa ? ak[u] : bk[v]);  // k left from this piece's start
    f32x8 o;
    if (isa ? AX : BX) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = inside || e < kl ? s[e * ld] : 0.f;
        if (e < 4) o.lo[e & 3] = x;
        else o.hi[e & 3] = x;
      }
    } else if (inside) {
      o = f32x8{*reinterpret_cast<const f32x4_u4*>(s), *reinterpret_cast<const f32x4_u4*>(s + 4)};
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = e < kl ? s[e] : 0.f;
        if (e < 4) o.lo[e & 3] = x;
        else o.hi[e & 3] = x;
      }
    }
    return o;
  };
  auto load = [&](int t, f32x8* q) {
    if (t >= NS) return;
    if (t < whole) {
#pragma unroll
      for (int w = 0; w < DA + DB; ++w) q[w] = load_piece(t, w, true);
    } else {
#pragma unroll
      for (int w = 0; w < DA + DB; ++w) q[w] = load_piece(t, w, false);
    }
  };

  // The products of the leading parts in one accumulator, the five smaller
  // ones in another: only one rounding per 32 k at the size of the result.
  f32x4 acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The six kept products, as (part of A, part of B).
  constexpr int QA[6] = {2, 1, 0, 1, 0, 0}, QB[6] = {0, 0, 0, 1, 1, 2};

  // The largest magnitude this thread has split of each piece's row (column).
  constexpr int W = DA + DB;
  float most[W];
#pragma unroll
  for (int w = 0; w < W; ++w) most[w] = 0.f;
  {
    const int af_off = frag_offset<BM, false>(wm * 16 * TM, lane);
    const int bf_off = 3 * APLANE + frag_offset<BN, false>(wn * 16 * TN, lane);
    u32x4 af[3][TM], bf[3][TN];
    auto read_a = [&](const unsigned char* st, int s, int q) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        af[q][i] = *reinterpret_cast<const u32x4*>(st + af_off + q * APLANE + s * 64 * BM + 1024 * i);
    };
    auto read_b = [&](const unsigned char* st, int s, int q) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bf[q][j] = *reinterpret_cast<const u32x4*>(st + bf_off + q * BPLANE + s * 64 * BN + 1024 * j);
    };
    auto product = [&](int g) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f32x4& c = g == 2 ? acc[i][j] : low[i][j];
          c = mfma16x16x32(bf[QB[g]][j], af[QA[g]][i], c);
        }
    };
    // Piece w of a step: its pair d of values into the three parts, and the
    // whole piece to LDS.
    u32x4 part[3];
    auto split_pair = [&](const f32x8& v, int w, int d) {
      const float x = d < 2 ? v.lo[2 * d] : v.hi[2 * d - 4], y = d < 2 ? v.lo[2 * d + 1] : v.hi[2 * d - 3];
      uint32_t p1, p2, p3;
      split2(x, y, p1, p2, p3);
      most[w] = fmaxf(most[w], fmaxf(fabsf(x), fabsf(y)));
      part[0][d] = p1;
      part[1][d] = p2;
      part[2][d] = p3;
    };
    auto put = [&](int slot, int w) {
      unsigned char* at = smem + slot * STEP + (w < DA ? aput[w < DA ? w : 0] : 3 * APLANE + bput[w < DA ? 0 : w - DA]);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(at + q * (w < DA ? APLANE : BPLANE)) = part[q];
    };
    auto store = [&](int slot, const f32x8* q) {
#pragma unroll
      for (int w = 0; w < W; ++w) {
#pragma unroll
        for (int d = 0; d < 4; ++d) split_pair(q[w], w, d);
        put(slot, w);
      }
    };
    if constexpr (KS == 1) {
      // Iteration t multiplies step t from registers.  As each fragment has
      // had its last use it is replaced by step t + 1's (LDS slot (t + 1) &
      // 1, complete since the barrier), two products or more before it is
      // needed; step t + 2, in registers, is split between the MFMAs into
      // slot t & 1, whose fragments every wave has had since the barrier,
      // and each of its pieces is followed by the load of step t + 3's.
      f32x8 q[W];
      load(0, q);
      store(0, q);
      load(1, q);
      if (NS > 1) store(1, q);
      load(2, q);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        read_a(smem, 0, r);
        read_b(smem, 0, r);
      }
      auto step = [&](auto inside, int t) {
        constexpr bool kInside = decltype(inside)::value;  // t + 3 < whole
        constexpr int NP = 4 * W;
        __syncthreads();
        const unsigned char* nx = smem + ((t + 1) & 1) * STEP;
        const bool more = kInside || t + 2 < NS;
#pragma unroll
        for (int g = 0; g < 6; ++g) {
          __builtin_amdgcn_sched_barrier(0);
          product(g);
          if (g == 0) read_a(nx, 0, 2);
          if (g == 2) read_b(nx, 0, 0);
          if (g == 3) read_a(nx, 0, 1);
          if (g == 4) read_b(nx, 0, 1);
          if (g == 5) {
            read_a(nx, 0, 0);
            read_b(nx, 0, 2);
          }
          if (more) {
#pragma unroll
            for (int e = g * NP / 6; e < (g + 1) * NP / 6; ++e) {
              split_pair(q[e / 4], e / 4, e % 4);
              if (e % 4 == 3) {
                put(t & 1, e / 4);
                if (kInside) q[e / 4] = load_piece(t + 3, e / 4, true);
              }
            }
          }
        }
        if (!kInside) load(t + 3, q);
      };
      int t = 0;
      for (; t + 3 < whole; ++t) step(std::true_type{}, t);
      for (; t < NS; ++t) step(std::false_type{}, t);
    } else {
      // Few rows: bound by the loads, two steps of which (in registers)
      // follow the one in LDS.
      f32x8 q[2][W];
      load(0, q[0]);
      load(1, q[1]);
      store(0, q[0]);
      load(2, q[0]);
      auto step = [&](auto parity, int t) {
        constexpr int P = decltype(parity)::value;  // t & 1
        __syncthreads();
        if (t + 1 < NS) store(P ^ 1, q[P ^ 1]);
        load(t + 3, q[P ^ 1]);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
          for (int r = 0; r < 3; ++r) {
            read_a(smem + P * STEP, s, r);
            read_b(smem + P * STEP, s, r);
          }
#pragma unroll
          for (int g = 0; g < 6; ++g) product(g);
        }
      };
      int t = 0;
      for (; t + 1 < NS; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
      }
      if (t < NS) step(std::integral_constant<int, 0>{}, t);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];

  // The results to recompute by f32 MFMAs (see above), a bit each.
  const int mloc = wm * 16 * TM + (lane & 15), nloc = wn * 16 * TN + 4 * (lane >> 4);
  auto line = [&](int w) { return w < DA ? ax[w < DA ? w : 0] : BM + bx[w < DA ? 0 : w - DA]; };
#pragma unroll
  for (int w = 0; w < W; ++w) atomicMax(big + line(w), __float_as_uint(most[w]));
  __syncthreads();
  static_assert(TM * TN * 4 <= 32, "a bit per result");
  const float kf = (float)K * kWholeTerms;
  // ranged: the smallest magnitudes are known (without them: every result
  // that is not kept for its own size, in a row and a column with a nonzero).
  auto doubtful = [&](auto ranged) {
    const float* bigf = reinterpret_cast<const float*>(big);
    const float* smallf = reinterpret_cast<const float*>(small);
    uint32_t bits = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const f32x4 bb = *reinterpret_cast<const f32x4*>(bigf + BM + nloc + 16 * j);
      f32x4 bs = {0.f, 0.f, 0.f, 0.f};
      if constexpr (ranged.value) bs = *reinterpret_cast<const f32x4*>(smallf + BM + nloc + 16 * j);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const float ab = bigf[mloc + 16 * i], as = ranged.value ? smallf[mloc + 16 * i] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float m = fabsf(acc[i][j][e]);
          if constexpr (ranged.value) asm volatile("" : "+v"(m));  // (nor from the first call to the second)
          bool keep = m >= kf * fmaxf(1.f, fmaxf(ab, bb[e])) || fminf(ab, bb[e]) == 0.f;
          if constexpr (ranged.value)
            keep = keep || (as * bs[e] >= kWholeTerms && fminf(as, bs[e]) >= kWholeParts);
          bits |= keep && m < __builtin_inff() ? 0u : 1u << (4 * (TM * j + i) + e);
        }
      }
    }
    asm volatile("" : "+v"(bits));  // (else each bit's condition is held to the end in registers of its own)
    return bits;
  };
  // Whether all of this lane's results are kept for their size, by one bound.
  auto all_large = [&] {
    const float* bigf = reinterpret_cast<const float*>(big);
    float most_of = 1.f;
    f32x4 least_of = {__builtin_inff(), __builtin_inff(), __builtin_inff(), __builtin_inff()};
    f32x4 zero = {0.f, 0.f, 0.f, 0.f};  // NaN after an infinity or a NaN
#pragma unroll
    for (int i = 0; i < TM; ++i) most_of = fmaxf(most_of, bigf[mloc + 16 * i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const f32x4 bb = *reinterpret_cast<const f32x4*>(bigf + BM + nloc + 16 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) most_of = fmaxf(most_of, bb[e]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          least_of[e] = fminf(least_of[e], fabsf(acc[i][j][e]));
          zero[e] = __builtin_fmaf(acc[i][j][e], 0.f, zero[e]);
        }
    }
    return zero.x + zero.y + zero.z + zero.w == 0.f &&
           fminf(fminf(least_of.x, least_of.y), fminf(least_of.z, least_of.w)) >= kf * most_of;
  };
  auto in_tile = [&](uint32_t bits) {
    if (bits) {
      flag[0] = 1;
      bool finite = false;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            finite |= (bits >> (4 * (TM * j + i) + e) & 1) && fabsf(acc[i][j][e]) < __builtin_inff();
      if (finite) flag[1] = 1;
    }
    __syncthreads();
  };
  uint32_t redo = all_large() ? 0u : doubtful(std::false_type{});
  in_tile(redo);
  if (flag[1]) {
    // Read the operands again for their smallest magnitudes, as twice their
    // bits less one (zero: ~0).
    uint32_t least[W];
#pragma unroll
    for (int w = 0; w < W; ++w) least[w] = ~0u;
    f32x8 q[W];
    load(0, q);
    for (int t = 0; t < NS; ++t) {
      f32x8 c[W];
#pragma unroll
      for (int w = 0; w < W; ++w) c[w] = q[w];
      if constexpr (KS == 1) load(t + 1, q);
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          least[w] = min(least[w], 2 * __float_as_uint(e < 4 ? c[w].lo[e & 3] : c[w].hi[e & 3]) - 1);
      if constexpr (KS > 1) load(t + 1, q);  // (its 128 k are in flight together already)
    }
#pragma unroll
    for (int w = 0; w < W; ++w)
      if (least[w] != ~0u) atomicMin(small + line(w), (least[w] >> 1) + 1);
    __syncthreads();
    if (tid == 0) flag[0] = 0;
    redo = doubtful(std::true_type{});
    __syncthreads();
    in_tile(redo);
  }
  if (flag[0]) {
    // f32 tiles in LDS (double buffered, loads a step ahead) and
    // v_mfma_f32_16x16x4_f32; in each 32 k, lane group g feeds k = 8g + s to
    // the s-th.  The sums go to `low`.
    constexpr int LD = BK + 4;  // floats
    static_assert(2 * (BM + BN) * LD * 4 <= 2 * STEP, "LDS");
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) low[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x8 q[W];
    load(0, q);
    for (int t = 0; t < NS; ++t) {
      float* fa = reinterpret_cast<float*>(smem) + (t & 1) * (BM + BN) * LD;
      float* fb = fa + BM * LD;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        float* d = w < DA ? fa + ax[w < DA ? w : 0] * LD + ak[w < DA ? w : 0]
                          : fb + bx[w < DA ? 0 : w - DA] * LD + bk[w < DA ? 0 : w - DA];
        *reinterpret_cast<f32x4*>(d) = q[w].lo;
        *reinterpret_cast<f32x4*>(d + 4) = q[w].hi;
      }
      __syncthreads();  // step t is whole, and every wave is done with step t - 1
      load(t + 1, q);
#pragma unroll 1
      for (int s = 0; s < KS; ++s) {
        const int k = 32 * s + 8 * (lane >> 4);
        f32x4 av[TM][2], bv[TN][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int i = 0; i < TM; ++i) av[i][h] = *reinterpret_cast<const f32x4*>(fa + (mloc + 16 * i) * LD + k + 4 * h);
#pragma unroll
          for (int j = 0; j < TN; ++j)
            bv[j][h] =
                *reinterpret_cast<const f32x4*>(fb + (wn * 16 * TN + (lane & 15) + 16 * j) * LD + k + 4 * h);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              low[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j][e >> 2][e & 3], av[i][e >> 2][e & 3], low[i][j],
                                                               0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[i][j][e] = redo >> (4 * (TM * j + i) + e) & 1 ? low[i][j][e] + 0.f : acc[i][j][e];  // (-0 by underflow: +0, whatever the padding)
  }

  // Epilogue (C^T fragments): this lane holds row m, columns n .. n + 3.
  float* C = p.c + (int64_t)blockIdx.z * p.sc;
  const int mrow = m0 + mloc, ncol = n0 + nloc;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = mrow + 16 * i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = ncol + 16 * j;
      float* c = C + (int64_t)m * N + n;
      if (n + 4 <= N) {
        *reinterpret_cast<f32x4_u4*>(c) = acc[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) c[e] = acc[i][j][e];
      }
    }
  }
}

}  // namespace mk

namespace mkg {
namespace {

template <int BM, int BN, int WM, int WN, int KS, bool AT, bool BT>
hipError_t launch(const mk::SplitArgs& p, int64_t batch, hipStream_t st) {
  constexpr size_t lds = (size_t)2 * 3 * (BM + BN) * 64 * KS + (BM + BN) * 8 + 8;
  static_assert(lds <= 160 * 1024, "LDS");
  const void* fn = (const void*)mk::gemm_split_kernel<BM, BN, WM, WN, KS, AT, BT>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int64_t tiles = (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  hipLaunchKernelGGL((mk::gemm_split_kernel<BM, BN, WM, WN, KS, AT, BT>),
                     dim3((unsigned)tiles, 1, (unsigned)batch), dim3(WM * WN * 64), lds, st, p);
  return hipGetLastError();
}

template <bool AT, bool BT>
hipError_t launch_order(const mk::SplitArgs& p, int64_t batch, int tile, hipStream_t st) {
  switch (tile) {
    case 16: return launch<16, 64, 1, 4, 4, AT, BT>(p, batch, st);
    case 64: return launch<64, 64, 2, 2, 1, AT, BT>(p, batch, st);
    default: return launch<128, 128, 2, 4, 1, AT, BT>(p, batch, st);
  }
}

}  // namespace

hipError_t split_launch(const SplitGemm& g, int tile, hipStream_t st) {
  mk::SplitArgs p;
  p.a = g.a;
  p.b = g.b;
  p.c = g.c;
  p.M = (int)g.M;
  p.N = (int)g.N;
  p.K = (int)g.K;
  p.lda = g.lda;
  p.ldb = g.ldb;
  p.sa = g.sa;
  p.sb = g.sb;
  p.sc = g.M * g.N;
  if (tile == 0) {
    // us per 32 k of one tile alone on the chip, with one on every CU, and
    // per tile and CU with several, measured at K = 4096 (gemm_tile.hip has
    // the same model): 16 rows x 4096 51 / 86 / 156 us with 16- / 64- /
    // 128-row tiles, 256 rows 209 / 90 / 156, 4096 rows 3144 / 970 / 711.
    struct Rate {
      int tile, bm, bn;
      double alone, full, each;
    };
    constexpr Rate kRates[3] = {{16, 16, 64, 0.39, 0.43, 0.385}, {64, 64, 64, 0.66, 0.70, 0.49},
                                {128, 128, 128, 1.20, 1.58, 1.39}};
    double least = 0;
    for (const Rate& r : kRates) {
      const int64_t tiles = ((g.M + r.bm - 1) / r.bm) * ((g.N + r.bn - 1) / r.bn);
      if (tiles * 512 > (int64_t)UINT32_MAX && r.tile != 128) continue;  // more threads than a launch has
      const double f = (double)((g.M + r.bm - 1) / r.bm) * (double)((g.N + r.bn - 1) / r.bn) * (double)g.batch / 256;
      const double t = f <= 1.0 ? r.alone + (r.full - r.alone) * f : std::max(r.full, std::ceil(f) * r.each);
      if (tile == 0 || t < least) {
        tile = r.tile;
        least = t;
      }
    }
  }
  switch ((g.a_t ? 2 : 0) + (g.b_t ? 1 : 0)) {
    case 0: return launch_order<false, false>(p, g.batch, tile, st);
    case 1: return launch_order<false, true>(p, g.batch, tile, st);
    case 2: return launch_order<true, false>(p, g.batch, tile, st);
    default: return launch_order<true, true>(p, g.batch, tile, st);
  }
}

}  // namespace mkg
