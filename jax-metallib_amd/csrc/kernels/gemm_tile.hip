// Tiled 16-bit GEMM of any size and operand order for gfx950 (MFMA
// 16x16x32, f32 accumulation).
//
// gemm.hip's 256 x 256 kernels need M and N in multiples of 256 and enough
// of those tiles to fill 256 CUs.  This family takes everything else: a
// decode step's 1..64 rows, ragged rows and columns, small products whose
// tiles must be small to reach every CU, operands stored transposed (a
// linear layer's dy W^T and x^T dy) and odd sizes.
//
//   * One kernel template over the tile (16 x 64 up to 256 x 256), the
//     storage order of each operand and how it is fed.
//   * An operand stored with k contiguous is staged as rows of 32 k (64
//     bytes; 16-byte chunk c of row r at c ^ (r / 2 % 4)) and read with
//     ds_read_b128; one stored with m or n contiguous is staged as k rows
//     and read with the transposing ds_read_b64_tr_b16.  The chunk swizzle
//     of the latter spreads the 8 k rows that a half wave reads at once over
//     all 64 banks for each row length (swz_x).
//   * Fed by LDS DMA through a ring of S steps of 32 KS k: no staging
//     registers, one barrier per step, (S - 1) steps in flight, which is
//     what the small tiles live on (16 x 64: 60 KB in flight per workgroup).
//     Pieces beyond K come from a zero page; rows and columns beyond M and N
//     repeat valid ones, whose results are not stored.  The main loop has no
//     branch per piece: with one, 256 rows of 4096 x 4096 on 64 x 64 tiles
//     took 22.6 us, without it 16.8, 128 x 128 tiles 37.7 and 29.6.
//   * 16-bit results go through LDS and leave in 16-byte pieces side by side
//     (1000 x 14336 x 4096 on 256 x 256 tiles, with the loop: 115 -> 102 us).
//   * Operands whose rows are not 16-byte aligned are fed through registers
//     (unaligned 16-byte loads, double-buffered LDS, the next step's loads
//     under this step's MFMAs).
//   * Every output accumulates its k in the order, and in the MFMA, that
//     gemm.hip's kernels use: the same bits as they give.
#include "common.h"
#include "epilogue.h"
#include "gemm_tile.h"
#include "gemm_tile_dev.h"

#include <math.h>

#include <type_traits>

namespace mk {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

struct TileArgs {
  const uint16_t* a;
  const uint16_t* b;
  void* c;
  const uint16_t* aux;
  int M, N, K;
  int64_t lda, ldb, sa, sb, sc;
  int64_t lima, limb;  // elements of one batch's operand that may be read
  int out_f32, epi;
  int narrow;  // an m- / n-contiguous operand with rows of fewer than 8 elements
};

// 16 bytes of zeros: the DMA source of pieces beyond K.
__device__ __align__(16) uint32_t g_tile_zero[4];

template <bool F16>
__device__ __forceinline__ f32x4 tile_mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  else
    return mfma16x16x32(a, b, c);
}

typedef u32x4 __attribute__((aligned(2))) u32x4_u2;
typedef u32x2 __attribute__((aligned(2))) u32x2_u2;
typedef f32x4 __attribute__((aligned(4))) f32x4_u4;

// Eight 16-bit elements at p + off, elements from lim on read as zero.
__device__ __forceinline__ u32x4 load8_lim(const uint16_t* p, int64_t off, int64_t lim) {
  if (off + 8 <= lim) return *reinterpret_cast<const u32x4_u2*>(p + off);
  uint32_t v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = off + e < lim ? (uint32_t)p[off + e] : 0u;
  return u32x4{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
}

// The first n (0..8) 16-bit elements kept, the rest zeroed.
__device__ __forceinline__ u32x4 keep8(const u32x4& v, int n) {
  u32x4 o;
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = v[d] & (n >= 2 * d + 2 ? 0xffffffffu : n == 2 * d + 1 ? 0xffffu : 0u);
  return o;
}

template <bool F16>
__device__ __forceinline__ u32x2 tile_pack4(const f32x4& v) {
  if constexpr (F16) {
    auto h = [](float f) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f); };
    return u32x2{h(v.x) | (h(v.y) << 16), h(v.z) | (h(v.w) << 16)};
  } else {
    return u32x2{pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
  }
}

// Eight consecutive 16-bit results of one row; the epilogues start from the
// rounded product, which is what v holds.
template <bool F16>
__device__ __forceinline__ void tile_store8(const TileArgs& p, int64_t zc, int m, int n, const u32x4& v) {
  const int64_t off = zc + (int64_t)m * p.N + n;
  uint16_t* c = static_cast<uint16_t*>(p.c) + off;
  if (!F16 && p.epi != MK_EPI_NONE) {  // N % 4 == 0
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (n + 4 * h >= p.N) break;
      const uint32_t a = v[2 * h], b = v[2 * h + 1];
      epi_store_bf16x4(static_cast<uint16_t*>(p.c), p.aux, p.epi, (size_t)(off + 4 * h),
                       f32x4{bf16_to_f32(a & 0xffffu), bf16_to_f32(a >> 16), bf16_to_f32(b & 0xffffu), bf16_to_f32(b >> 16)});
    }
  } else if (n + 8 <= p.N) {
    *reinterpret_cast<u32x4_u2*>(c) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (n + e < p.N) c[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
  }
}

// Four consecutive f32 results of one row.
__device__ __forceinline__ void tile_store4(const TileArgs& p, int64_t zc, int m, int n, const f32x4& v) {
  float* c = static_cast<float*>(p.c) + zc + (int64_t)m * p.N + n;
  if (n + 4 <= p.N) {
    *reinterpret_cast<f32x4_u4*>(c) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) c[e] = v[e];
  }
}

template <int BM, int BN, int WM, int WN, int KS, int S, bool AT, bool BT, bool F16, bool DMA>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_tile_kernel(TileArgs p) {
  constexpr int NW = WM * WN, BK = 32 * KS;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int IA = KS * BM / 16, IB = KS * BN / 16;  // 1 KB pieces of a step
  constexpr int DA = IA / NW, DB = IB / NW;            // per wave
  static_assert(DA * NW == IA && DB * NW == IB, "the waves share the pieces evenly");
  constexpr int ABYTES = IA * 1024, STEP = (IA + IB) * 1024;
  constexpr bool AX = AT, BX = !BT;  // the operand's m / n is contiguous

  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int M = p.M, N = p.N, K = p.K;
  int m0, n0;
  tile_origin(M, N, BM, BN, m0, n0);
  const uint16_t* A = p.a + (int64_t)blockIdx.z * p.sa;
  const uint16_t* B = p.b + (int64_t)blockIdx.z * p.sb;

  // This lane's source element of each piece (step 0) and its k.
  int64_t aoff[DA], boff[DB];
  int ak[DA], bk[DB];
#pragma unroll
  for (int u = 0; u < DA; ++u) {
    int x;
    stage_coord<BM, AX>(DA * wave + u, lane, x, ak[u]);
    x += m0;
    if (AX) aoff[u] = (int64_t)ak[u] * p.lda + (x < M ? x : 0);
    else aoff[u] = (int64_t)(x < M ? x : M - 1) * p.lda + ak[u];
  }
#pragma unroll
  for (int u = 0; u < DB; ++u) {
    int x;
    stage_coord<BN, BX>(DB * wave + u, lane, x, bk[u]);
    x += n0;
    if (BX) boff[u] = (int64_t)bk[u] * p.ldb + (x < N ? x : 0);
    else boff[u] = (int64_t)(x < N ? x : N - 1) * p.ldb + bk[u];
  }
  const int64_t astep = AX ? (int64_t)BK * p.lda : BK, bstep = BX ? (int64_t)BK * p.ldb : BK;

  // Fragment offsets within a step.
  int af_off[AX ? TM : 1], bf_off[BX ? TN : 1];
#pragma unroll
  for (int i = 0; i < (AX ? TM : 1); ++i) af_off[i] = frag_offset<BM, AX>(wm * 16 * TM + 16 * i, lane);
#pragma unroll
  for (int j = 0; j < (BX ? TN : 1); ++j) bf_off[j] = ABYTES + frag_offset<BN, BX>(wn * 16 * TN + 16 * j, lane);

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int NS = (K + BK - 1) / BK;
  const bool ragged = K % BK != 0;
  if constexpr (DMA) {
    const uint32_t sbase = lds_addr(smem);
    const uint16_t *ap[DA], *bp[DB];
#pragma unroll
    for (int u = 0; u < DA; ++u) ap[u] = A + aoff[u];
#pragma unroll
    for (int u = 0; u < DB; ++u) bp[u] = B + boff[u];
    // Piece u of the next step into the slot at st; the steps are issued in
    // order, so each pointer advances by one step.
    constexpr int D = DA + DB;
    auto issue = [&](uint32_t st, int u) {
      if (u < DA) {
        dma16_asm(ap[u < DA ? u : 0], st + (uint32_t)((DA * wave + u) * 1024));
        ap[u < DA ? u : 0] += astep;
      } else {
        const int v = u < DA ? 0 : u - DA;
        dma16_asm(bp[v], st + (uint32_t)(ABYTES + (DB * wave + v) * 1024));
        bp[v] += bstep;
      }
    };
    // Before the last step when K ends inside it: pieces beyond K read zeros.
    auto cut_k = [&](int t) {
      if (ragged && t == NS - 1) {
        const uint16_t* z = reinterpret_cast<const uint16_t*>(g_tile_zero);
#pragma unroll
        for (int u = 0; u < DA; ++u) ap[u] = t * BK + ak[u] < K ? ap[u] : z;
#pragma unroll
        for (int u = 0; u < DB; ++u) bp[u] = t * BK + bk[u] < K ? bp[u] : z;
      }
    };
    auto read_a = [&](const unsigned char* st, int s, int i) {
      return read_frag<BM, AX>(st + s * 64 * BM + (AX ? af_off[AX ? i : 0] : af_off[0] + 1024 * i));
    };
    auto read_b = [&](const unsigned char* st, int s, int j) {
      return read_frag<BN, BX>(st + s * 64 * BN + (BX ? bf_off[BX ? j : 0] : bf_off[0] + 1024 * j));
    };
    const int pre = NS < S ? NS : S;
    for (int t = 0; t < pre; ++t) {
      cut_k(t);
#pragma unroll
      for (int u = 0; u < D; ++u) issue(sbase + (uint32_t)(t * STEP), u);
    }
    if (NS >= S) vm_wait(D * (S - 1));
    else vm_wait(0);
    asm volatile("s_barrier" ::: "memory");
    // Fragments are read one 32-k part ahead of the MFMAs that use them: B
    // in two register sets, A's fragment i into the registers of the part
    // before right after their last MFMA.
    u32x4 af[TM], bf[2][TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[0][j] = read_b(smem, 0, j);
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = read_a(smem, 0, i);
    int slot = 0;  // slot of step t
    // ALWAYS: step t + S exists, whole, and is issued during this one's last
    // part (no branch per piece: the main loop).
    auto step = [&](auto parity, auto always, int t) {
      constexpr int P = decltype(parity)::value;
      constexpr bool ALWAYS = decltype(always)::value;
      const bool more = ALWAYS || t + S < NS;
      const unsigned char* cur = smem + slot * STEP;
      const int slot_nx = slot + 1 == S ? 0 : slot + 1;
      const unsigned char* nxt = smem + slot_nx * STEP;
      const uint32_t fill = sbase + (uint32_t)(slot * STEP);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bool lastpart = s == KS - 1;
        if (lastpart) {
          __builtin_amdgcn_sched_barrier(0);
          // This wave's pieces of step t + 1 have landed and its fragments
          // of step t are in registers; past the barrier that is so for
          // every wave: step t + 1 may be read, step t's slot refilled.
          // (After the last step the reads below take a stale slot; their
          // values are not used.)
          if (ALWAYS || t + S - 1 < NS) vm_wait(D * (S - 2));
          else vm_wait(0);
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
          if (!ALWAYS && more) cut_k(t + S);
        }
        const unsigned char* from = lastpart ? nxt : cur;
        const int sn = lastpart ? 0 : s + 1;
        const int c = (P + s) & 1;  // folds: s is unrolled
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[c ^ 1][j] = read_b(from, sn, j);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = tile_mfma<F16>(bf[c][j], af[i], acc[i][j]);
          af[i] = read_a(from, sn, i);
          if (lastpart && more) {
#pragma unroll
            for (int u = i * D / TM; u < (i + 1) * D / TM; ++u) issue(fill, u);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      slot = slot_nx;
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, KS % 2>;  // B's register sets turn over KS times a step
    int t = 0;
    for (; t + 2 + S < NS; t += 2) {
      step(I0{}, std::true_type{}, t);
      step(I1{}, std::true_type{}, t + 1);
    }
    for (; t + 1 < NS; t += 2) {
      step(I0{}, std::false_type{}, t);
      step(I1{}, std::false_type{}, t + 1);
    }
    if (t < NS) step(I0{}, std::false_type{}, t);
  } else {
    auto multiply = [&](const unsigned char* st) {
  #pragma unroll
      for (int s = 0; s < KS; ++s) {
        u32x4 bf[TN];
  #pragma unroll
        for (int j = 0; j < TN; ++j)
          bf[j] = read_frag<BN, BX>(st + s * 64 * BN + (BX ? bf_off[BX ? j : 0] : bf_off[0] + 1024 * j));
  #pragma unroll
        for (int i = 0; i < TM; ++i) {
          const u32x4 af = read_frag<BM, AX>(st + s * 64 * BM + (AX ? af_off[AX ? i : 0] : af_off[0] + 1024 * i));
  #pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = tile_mfma<F16>(bf[j], af, acc[i][j]);
        }
      }
    };
    // Registers hold two steps ahead of the one being multiplied: set t & 1
    // takes step t's loads two iterations before they go to LDS.
    u32x4 ra[2][DA], rb[2][DB];
    auto load = [&](int t, u32x4* qa, u32x4* qb) {
      if (t >= NS) return;
      const int64_t at = t * astep, bt = t * bstep;
      if (t < NS - 1 && !p.narrow) {  // every piece inside the operands
#pragma unroll
        for (int u = 0; u < DA; ++u) qa[u] = *reinterpret_cast<const u32x4_u2*>(A + aoff[u] + at);
#pragma unroll
        for (int u = 0; u < DB; ++u) qb[u] = *reinterpret_cast<const u32x4_u2*>(B + boff[u] + bt);
        return;
      }
      const int kl = K - t * BK;  // k left from this step's start
#pragma unroll
      for (int u = 0; u < DA; ++u)
        qa[u] = ak[u] < kl ? load8_lim(A, aoff[u] + at, p.lima) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int u = 0; u < DB; ++u)
        qb[u] = bk[u] < kl ? load8_lim(B, boff[u] + bt, p.limb) : u32x4{0u, 0u, 0u, 0u};
      // A piece along k may run past K into the next row.
      if constexpr (!AX) {
#pragma unroll
        for (int u = 0; u < DA; ++u) qa[u] = keep8(qa[u], kl - ak[u]);
      }
      if constexpr (!BX) {
#pragma unroll
        for (int u = 0; u < DB; ++u) qb[u] = keep8(qb[u], kl - bk[u]);
      }
    };
    auto store = [&](int slot, const u32x4* qa, const u32x4* qb) {
      unsigned char* st = smem + slot * STEP + 16 * lane;
#pragma unroll
      for (int u = 0; u < DA; ++u) *reinterpret_cast<u32x4*>(st + (DA * wave + u) * 1024) = qa[u];
#pragma unroll
      for (int u = 0; u < DB; ++u) *reinterpret_cast<u32x4*>(st + ABYTES + (DB * wave + u) * 1024) = qb[u];
    };
    load(0, ra[0], rb[0]);
    load(1, ra[1], rb[1]);
    store(0, ra[0], rb[0]);
    load(2, ra[0], rb[0]);
    // Step t is in LDS slot t & 1; its barrier also says that every wave is
    // done with step t - 1, whose slot step t + 1 (in registers) takes.
    auto step = [&](auto parity, int t) {
      constexpr int P = decltype(parity)::value;  // t & 1
      __syncthreads();
      if (t + 1 < NS) store(P ^ 1, ra[P ^ 1], rb[P ^ 1]);
      load(t + 3, ra[P ^ 1], rb[P ^ 1]);
      multiply(smem + P * STEP);
    };
    int t = 0;
    for (; t + 1 < NS; t += 2) {
      step(std::integral_constant<int, 0>{}, t);
      step(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < NS) step(std::integral_constant<int, 0>{}, t);
  }

  // Epilogue (C^T fragments): this lane holds row m, columns n .. n + 3.
  const int64_t zc = (int64_t)blockIdx.z * p.sc;
  if (!p.out_f32) {
    // 16-bit results through LDS, so that a row leaves in 16-byte pieces side
    // by side; the row padding spreads the writes over all banks.
    constexpr int RS = BN + 16;
    uint16_t* stage = reinterpret_cast<uint16_t*>(smem);
    __syncthreads();  // every wave is done with the ring
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *reinterpret_cast<u32x2*>(stage + (wm * 16 * TM + 16 * i + (lane & 15)) * RS + wn * 16 * TN + 16 * j +
                                  4 * (lane >> 4)) = tile_pack4<F16>(acc[i][j]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < (BM * BN / 8 + NW * 64 - 1) / (NW * 64); ++q) {
      const int c = q * NW * 64 + tid, row = c / (BN / 8), col = 8 * (c % (BN / 8));
      if (BM * BN / 8 < NW * 64 && row >= BM) break;  // the smallest tile has fewer pieces than threads
      if (m0 + row < M && n0 + col < N)
        tile_store8<F16>(p, zc, m0 + row, n0 + col, *reinterpret_cast<const u32x4*>(stage + row * RS + col));
    }
    return;
  }
  const int mrow = m0 + wm * 16 * TM + (lane & 15), ncol = n0 + wn * 16 * TN + 4 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = mrow + 16 * i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = ncol + 16 * j;
      if (n < N) tile_store4(p, zc, m, n, acc[i][j]);
    }
  }
}

}  // namespace mk

namespace mkg {
namespace {

constexpr int kCus = 256;

constexpr int step_bytes(int bm, int bn, int ks) { return (bm + bn) * 64 * ks; }

template <int BM, int BN, int WM, int WN, int KS, int S, bool AT, bool BT, bool F16, bool DMA>
hipError_t launch(const mk::TileArgs& p, int64_t batch, hipStream_t st) {
  constexpr size_t ring = (size_t)S * step_bytes(BM, BN, KS), stage = (size_t)BM * (BN + 16) * 2;
  constexpr size_t lds = ring > stage ? ring : stage;
  static_assert(lds <= 160 * 1024, "LDS");
  const void* fn = (const void*)mk::gemm_tile_kernel<BM, BN, WM, WN, KS, S, AT, BT, F16, DMA>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int64_t tiles = (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  hipLaunchKernelGGL((mk::gemm_tile_kernel<BM, BN, WM, WN, KS, S, AT, BT, F16, DMA>),
                     dim3((unsigned)tiles, 1, (unsigned)batch), dim3(WM * WN * 64), lds, st, p);
  return hipGetLastError();
}

// DMA-fed: all six shapes.
template <bool AT, bool BT>
hipError_t launch_dma(const mk::TileArgs& p, int64_t batch, int shape, hipStream_t st) {
  switch (shape) {
    case T16x64: return launch<16, 64, 1, 4, 4, 3, AT, BT, false, true>(p, batch, st);
    case T32x64: return launch<32, 64, 1, 4, 4, 3, AT, BT, false, true>(p, batch, st);
    case T64x64: return launch<64, 64, 2, 2, 2, 4, AT, BT, false, true>(p, batch, st);
    case T128x64: return launch<128, 64, 2, 2, 2, 3, AT, BT, false, true>(p, batch, st);
    case T128x128:
      // A workgroup alone on its CU needs two steps in flight (96 KB of
      // LDS); with more tiles than CUs two workgroups of one step each
      // cover for one another.  Two steps / one: 2048^3 (256 tiles) 19.8 /
      // 24.9 us, 2000 x 3000 x 2048 (384) 35.2 / 30.0, 4096^3 151 / 133.
      if ((int64_t)((p.M + 127) / 128) * ((p.N + 127) / 128) * batch <= kCus)
        return launch<128, 128, 2, 2, 2, 3, AT, BT, false, true>(p, batch, st);
      return launch<128, 128, 2, 2, 2, 2, AT, BT, false, true>(p, batch, st);
    default: return launch<256, 256, 2, 4, 1, 5, AT, BT, false, true>(p, batch, st);
  }
}

// Fed through registers: three shapes.  f16 has these only: such products come
// from dot_general alone, and the DMA-fed instances, most of this file's code,
// are bf16's.
template <bool AT, bool BT, bool F16>
hipError_t launch_reg(const mk::TileArgs& p, int64_t batch, int shape, hipStream_t st) {
  switch (shape) {
    case T16x64: return launch<16, 64, 1, 4, 4, 2, AT, BT, F16, false>(p, batch, st);
    case T32x64:
    case T64x64: return launch<64, 64, 2, 2, 2, 2, AT, BT, F16, false>(p, batch, st);
    default: return launch<128, 128, 2, 4, 1, 2, AT, BT, F16, false>(p, batch, st);
  }
}

constexpr int kBm[kTileShapes] = {16, 32, 64, 128, 128, 256};
constexpr int kBn[kTileShapes] = {64, 64, 64, 64, 128, 256};

// us per 32 k of one tile: alone on the chip, with one on every CU, and per
// tile and CU with several (two resident).  Measured at K = 4096, e.g. fed by
// DMA, M x 4096: 16 rows 12.2 us (16 x 64; 64 x 64 13.9, 128 x 128 28.0),
// 128 rows 13.8 (32 x 64; 16 x 64 21.4), 256 rows 16.8 (64 x 64; 32 x 64
// 24.6, 128 x 64 21.5), 512 rows 25.1 (128 x 64; 64 x 64 32.2), 2000 rows
// 59.9 (128 x 128; 128 x 64 77.1, 256 x 256 87.6), 4096 rows 105.2 (256 x
// 256; 128 x 128 119.3).  Through registers (N = 4097): 16 rows 18.2 / 28.9 /
// 50.0 (16 x 64 / 64 x 64 / 128 x 128), 512 rows 117 / 59.7 / 54.8.
struct Rate {
  double alone, full, each;
};
constexpr Rate kDmaRate[kTileShapes] = {{0.088, 0.095, 0.060}, {0.094, 0.100, 0.075}, {0.101, 0.123, 0.112},
                                        {0.142, 0.188, 0.165}, {0.210, 0.280, 0.235}, {0.590, 0.790, 0.790}};
constexpr Rate kRegRate[kTileShapes] = {{0.148, 0.155, 0.109}, {1e9, 1e9, 1e9}, {0.225, 0.240, 0.175},
                                        {1e9, 1e9, 1e9}, {0.400, 0.490, 0.370}, {1e9, 1e9, 1e9}};
// us a CU spends on a tile besides: the first step's latency and the stores,
// half hidden where two workgroups share the CU.
constexpr double kTileOver[kTileShapes] = {0.1, 0.2, 0.3, 0.6, 1.2, 5.5};

}  // namespace

bool tile_grid_fits(int64_t M, int64_t N, int shape) {
  // 256 threads a tile fed by DMA (512: 256 x 256); through registers the
  // middle shapes are 64 x 64 tiles of 256 and the large ones 128 x 128 of 512.
  auto fits = [&](int64_t bm, int64_t bn, int64_t threads) {
    return ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * threads <= (int64_t)UINT32_MAX;
  };
  return fits(kBm[shape], kBn[shape], shape == T256x256 ? 512 : 256) && (shape < T128x64 || fits(128, 128, 512));
}

bool tile_dma_ok(const TileGemm& g) {
  if (g.f16 || g.registers) return false;
  auto ok = [&](const void* q, int64_t ld, int64_t s, int64_t contiguous) {
    return ((uintptr_t)q & 15) == 0 && ld % 8 == 0 && (g.batch == 1 || s % 8 == 0) && contiguous % 8 == 0;
  };
  return ok(g.a, g.lda, g.sa, g.a_t ? g.M : g.K) && ok(g.b, g.ldb, g.sb, g.b_t ? g.K : g.N);
}

double tile_estimate(const TileGemm& g, int shape) {
  const Rate& r = (tile_dma_ok(g) ? kDmaRate : kRegRate)[shape];
  const double f = (double)((g.M + kBm[shape] - 1) / kBm[shape]) * (double)((g.N + kBn[shape] - 1) / kBn[shape]) *
                   (double)g.batch / kCus;
  const double per32 = f <= 1.0 ? r.alone + (r.full - r.alone) * f : fmax(r.full, ceil(f) * r.each);
  return (double)((g.K + 31) / 32) * per32 + ceil(f) * kTileOver[shape] * (g.out_f32 ? 2.0 : 1.0);
}

int tile_pick(const TileGemm& g) {
  int best = -1;
  double cost = 0;
  for (int s = 0; s < kTileShapes; ++s) {
    if (!tile_grid_fits(g.M, g.N, s)) continue;
    const double c = tile_estimate(g, s);
    if (best < 0 || c < cost) {
      best = s;
      cost = c;
    }
  }
  return best < 0 ? T256x256 : best;
}

hipError_t tile_launch(const TileGemm& g, int shape, hipStream_t st) {
  mk::TileArgs p;
  p.a = static_cast<const uint16_t*>(g.a);
  p.b = static_cast<const uint16_t*>(g.b);
  p.c = g.c;
  p.aux = static_cast<const uint16_t*>(g.aux);
  p.M = (int)g.M;
  p.N = (int)g.N;
  p.K = (int)g.K;
  p.lda = g.lda;
  p.ldb = g.ldb;
  p.sa = g.sa;
  p.sb = g.sb;
  p.sc = g.M * g.N;
  p.lima = g.a_t ? (g.K - 1) * g.lda + g.M : (g.M - 1) * g.lda + g.K;
  p.limb = g.b_t ? (g.N - 1) * g.ldb + g.K : (g.K - 1) * g.ldb + g.N;
  p.out_f32 = g.out_f32 ? 1 : 0;
  p.epi = g.epi;
  p.narrow = (g.a_t && g.lda < 8) || (!g.b_t && g.ldb < 8);
  const int order = (g.a_t ? 2 : 0) + (g.b_t ? 1 : 0);
  if (tile_dma_ok(g)) {
    switch (order) {
      case 0: return launch_dma<false, false>(p, g.batch, shape, st);
      case 1: return launch_dma<false, true>(p, g.batch, shape, st);
      case 2: return launch_dma<true, false>(p, g.batch, shape, st);
      default: return launch_dma<true, true>(p, g.batch, shape, st);
    }
  }
#define MK_TILE_REG(F16)                                                   \
  switch (order) {                                                         \
    case 0: return launch_reg<false, false, F16>(p, g.batch, shape, st);   \
    case 1: return launch_reg<false, true, F16>(p, g.batch, shape, st);    \
    case 2: return launch_reg<true, false, F16>(p, g.batch, shape, st);    \
    default: return launch_reg<true, true, F16>(p, g.batch, shape, st);    \
  }
  if (g.f16) MK_TILE_REG(true)
  MK_TILE_REG(false)
#undef MK_TILE_REG
}

}  // namespace mkg
