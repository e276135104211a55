// Quantized matmul for a middling number of rows (17 to a thousand; fewer
// where K keeps the decode kernels out) on gfx950: y[M, N] = x[M, K] @
// dequant(W)[K, N], formats as in qmatmul.hip.
//
// The decode kernels there take 16 rows a pass and so convert the weights
// M / 16 times; the kernel of qgemm.hip pads to 256 rows and fills the chip
// with large N only.  Here a workgroup owns 32 to 128 rows x 128 columns and
// 1/ks of K, each weight is fetched and converted once per tile, and tile
// height and K split are chosen so that the grid is one or two rounds of the
// 256 CUs.
//
//   * x (bf16) and the packed weights come by LDS DMA through a ring of 64-k
//     steps, 128 KB or more per CU: the weights come from HBM, and that much
//     has to be in flight.
//   * KW groups of four waves take alternate steps, so that a SIMD has two
//     (four at BM = 32) waves and one's conversions run under the other's
//     MFMAs; with one wave a SIMD int8 at M = 100, K = 4096, N = 14336 took
//     35.2 us, with two 26.1, and with the conversions spread between the
//     MFMAs, half a step ahead of their use, 22.1.  A wave's tile is all rows
//     x 32 columns: it converts only weights that no other wave needs.  Every
//     wave reads all of x from LDS, and a transposing read costs twice its
//     bytes: int4 at 256 rows keeps LDS 1.3 times as busy as the 4096^3 GEMM
//     does, which LDS bounds (SQ_LDS_IDX_ACTIVE over the kernel's cycles), with
//     the MFMAs at 0.25.  int8 at 100 rows saturates nothing: LDS at 0.6 of
//     that, MFMAs 0.21, 2.5 TB/s, and waits for steps the rest of the time.
//   * Weights leave LDS by ds_read_b64_tr_b8: a lane gets 8 bytes of its
//     column, 8 k of int8 or 16 of int4.
//   * int8: the bytes as bf16 (exact), the column's scale on the f32 sum.
//     int4: q - z as bf16 (exact), each 64-k group summed by itself and
//     multiplied by its scale in f32: nothing is rounded before the store
//     (relative error 1.66e-3 against float64, that of the final rounding).
//   * ks > 1: as in qgemm.hip, f32 partials by device-coherent stores, an
//     arrival counter per tile, and the last arriver adds them in k order.
//
// K = 4096, N = 14336, us (before; the floor is the weights' 58.7 or 33 MB):
//   rows     17         64         100        256        700        1000
//   int8  16.6 (20)  18.6 (37)  22.2 (66)  32.6 (46)  91 (131)   121 (132)
//   int4  18.0 (19)  23.3 (34)  28.2 (57)  41.5 (46)  120 (128)  --
#include "common.h"
#include "epilogue.h"
#include "gemm_tile_dev.h"
#include "qtile.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace mk {

struct QTileArgs {
  const uint16_t* x;
  const uint8_t* w;
  const void* s;
  const uint8_t* z;
  uint16_t* y;
  const uint16_t* aux;
  int epi;
  int M, K, N, ks;
  float* part;    // [tile][ks][BM * 128] f32
  uint32_t* cnt;  // per-tile arrival counters (zero between calls)
};

constexpr int kQtCols = 128;

typedef int qt_i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) qt_i32x2* lds_qt_ptr;

__device__ __forceinline__ u32x2 read_tr8(const unsigned char* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_qt_ptr)(p)));
}

// LDS DMA of 16 (4) bytes a lane from base + off to lds_base + 16 (4) * lane
// (the s_nop: see dma16_asm).
__device__ __forceinline__ void dma16_sbase(const void* base, uint32_t off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_base)
               : "m0", "memory");
}

__device__ __forceinline__ void dma4_sbase(const void* base, uint32_t off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds_base)
               : "m0", "memory");
}

// 4-byte LDS DMA of every lane to lds_base + 4 * lane (see dma16_asm).
__device__ __forceinline__ void dma4_asm(const void* src, uint32_t lds_base) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(base)
               : "m0", "memory");
}

// Signed bytes 2d and 2d + 1 of w -> a pair of bf16, exactly.
__device__ __forceinline__ uint32_t int8_pair(const u32x2& w, int d) {
  const uint32_t v = d < 2 ? w.x : w.y;
  const int sh = 16 * (d & 1);
  return pack_bf16x2((float)(int8_t)(v >> sh), (float)(int8_t)(v >> (sh + 8)));
}

// d = half h of the f16 pair a, plus b, in f32.
template <int H>
__device__ __forceinline__ float half_plus(uint32_t a, float b) {
  float d;
  if constexpr (H == 0)
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(a), "v"(b));
  else
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(a), "v"(b));
  return d;
}

// Byte d of t (low nibble even k) minus the zero point -> a pair of bf16,
// exactly: a low nibble q in the f16 0x6400 + q is 1024 + q, a high one in
// 0x5400 + 16 q is 64 + q; nlo = -1024 - z and nhi = -64 - z take it to q - z
// in f32.
__device__ __forceinline__ uint32_t int4_pair(uint32_t t, int d, float nlo, float nhi) {
  const uint32_t u = d & 1 ? t >> 8 : t;
  const uint32_t lo = (u & 0x000F000Fu) | 0x64006400u, hi = (u & 0x00F000F0u) | 0x54005400u;
  return d < 2 ? pack_bf16x2(half_plus<0>(lo, nlo), half_plus<0>(hi, nhi))
               : pack_bf16x2(half_plus<1>(lo, nlo), half_plus<1>(hi, nhi));
}

// KW groups of four waves, each with a ring of S 64-k steps.  NARROW: N is a
// multiple of 8 only, so weight rows are 8-byte aligned and come 4 bytes a lane.
template <bool INT4, int BM, int S, int KW, bool NARROW>
__global__ __launch_bounds__(256 * KW) void qtile_kernel(QTileArgs p) {
  constexpr int TM = BM / 16, TN = 2, NW = 4;
  constexpr int ABYTES = BM * 128;                  // [BM rows][64 k] bf16
  constexpr int BROWS = INT4 ? 32 : 64;             // weight rows of a step
  constexpr int BBYTES = BROWS * kQtCols;
  constexpr int ZBYTES = INT4 ? NW * 256 : 0;       // each wave's scales and zero points
  constexpr int STEP = ABYTES + BBYTES + ZBYTES;
  constexpr int WPIECE = NARROW ? 256 : 1024;  // bytes of a weight piece
  constexpr int DA = ABYTES / 1024 / NW, DB = BBYTES / WPIECE / NW, D = DA + DB + (INT4 ? 1 : 0);
  static_assert(DA * NW * 1024 == ABYTES && S * KW * STEP <= 160 * 1024 && KW * BM * kQtCols * 4 <= 160 * 1024 && D * (S - 1) <= 63, "ring");

  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int M = p.M, N = p.N, K = p.K;
  const int tiles_m = (M + BM - 1) / BM;
  const int L = xcd_run_id(blockIdx.x, gridDim.x);
  const int tile = L / p.ks, ksi = L - tile * p.ks;
  const int tn = tile / tiles_m, m0 = (tile - tn * tiles_m) * BM, n0 = tn * kQtCols;
  const int n0w = n0 + 32 * wave;  // this wave's columns
  // This part's 64-k steps.
  const int groups = K / 64, gb = (int)((int64_t)groups * ksi / p.ks);
  const int gn = (int)((int64_t)groups * (ksi + 1) / p.ks) - gb;
  // Wave group kw takes steps kw, kw + KW, ...: NS of them from k group g0,
  // one fewer than NT where they do not come out even.
  const int g0 = gb + kw, NS = (gn - kw + KW - 1) / KW, NT = (gn + KW - 1) / KW;

  // DMA sources.  x piece q: rows 8q .. 8q + 7, 16-byte chunk c of row r at
  // c ^ (r & 7).  Weight piece q: rows 8q .. 8q + 7 of 128 bytes, 16-column
  // chunk c of row r at c ^ ((r / 2) % 8).  A lane's offset is the same every
  // step; the scalar bases advance.  (NARROW: piece q is rows 2q, 2q + 1 in
  // the same layout.)
  const uint16_t* abase = p.x + (int64_t)m0 * K + 64 * g0;
  const uint8_t* bbase = p.w + (int64_t)g0 * BROWS * N;
  uint32_t aof[DA], bof[DB];
#pragma unroll
  for (int u = 0; u < DA; ++u) {
    const int r = 8 * (DA * wave + u) + (lane >> 3), c = (lane & 7) ^ (r & 7);
    aof[u] = 2 * ((uint32_t)min(r, M - 1 - m0) * (uint32_t)K + 8u * c);
  }
#pragma unroll
  for (int u = 0; u < DB; ++u) {
    if constexpr (NARROW) {
      const int r = 2 * (DB * wave + u) + (lane >> 5), c = ((lane >> 2) & 7) ^ ((r >> 1) & 7);
      bof[u] = (uint32_t)r * (uint32_t)N + (uint32_t)min(n0 + 16 * c + 4 * (lane & 3), N - 4);
    } else {
      const int r = 8 * (DB * wave + u) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      bof[u] = (uint32_t)r * (uint32_t)N + (uint32_t)min(n0 + 16 * c, N - 16);
    }
  }
  // int4: lanes 0-15 this wave's 32 scales, 16-23 its zero points.
  const unsigned char* zp = nullptr;
  int64_t zstep = 0;
  if constexpr (INT4) {
    if (lane >= 16 && lane < 24) {
      zp = p.z + (int64_t)g0 * N + min(n0w + 4 * (lane - 16), N - 4);
      zstep = KW * N;
    } else {
      zp = reinterpret_cast<const unsigned char*>(static_cast<const uint16_t*>(p.s) + (int64_t)g0 * N +
                                                  min(n0w + 2 * (lane & 15), N - 2));
      zstep = 2 * KW * (int64_t)N;
    }
  }
  unsigned char* const ring = smem + kw * (S * STEP);
  const uint32_t sbase = lds_addr(ring);
  // Piece u of the next step into the ring slot at `st`.
  auto issue = [&](uint32_t st, int u) {
    if (u < DA) dma16_sbase(abase, aof[u < DA ? u : 0], st + (uint32_t)((DA * wave + u) * 1024));
    else if (u < DA + DB)
      (NARROW ? dma4_sbase : dma16_sbase)(bbase, bof[u < DA || u >= DA + DB ? 0 : u - DA],
                                          st + (uint32_t)(ABYTES + (DB * wave + u - DA) * WPIECE));
    else dma4_asm(zp, st + (uint32_t)(ABYTES + BBYTES + 256 * wave));
  };
  auto advance = [&]() {
    abase += 64 * KW;
    bbase += (int64_t)(BROWS * KW) * N;
    if constexpr (INT4) zp += zstep;
  };

  // Fragment addresses.  x: row 16 i + lane % 16, chunk 4h + g (int8: k = 32
  // h + 8 g) or 2g + h (int4: k = 16 g + 8 h), g = lane / 16.  Weights: the
  // transposing read of lane group g takes rows 8g .. 8g + 7 (int8: + 32 h).
  const int g4 = lane >> 4;
  int aoff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) aoff[h] = (lane & 15) * 128 + 16 * ((INT4 ? 2 * g4 + h : 4 * h + g4) ^ (lane & 7));
  const int brow = 8 * g4 + ((lane & 15) >> 1);
  int boff[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    boff[j] = ABYTES + brow * kQtCols + 16 * ((2 * wave + j) ^ ((brow >> 1) & 7)) + 8 * (lane & 1);
  const int zoff = ABYTES + BBYTES + 256 * wave;

  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TM][TN], y[INT4 ? TM : 1][INT4 ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = zero4;
      if constexpr (INT4) y[i][j] = zero4;
    }

  // af, bf[0] and `raw` hold step t at the head of its loop pass.
  u32x4 af[2][TM], bf[2][TN];
  struct Raw {
    u32x2 w[INT4 ? TN : 2 * TN], s[TN];
    uint32_t z[TN];
  } raw;
  auto read_a = [&](const unsigned char* st, int h, int i) {
    af[h][i] = *reinterpret_cast<const u32x4*>(st + aoff[h] + 2048 * i);
  };
  auto read_raw = [&](const unsigned char* st, Raw& r) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (INT4) {
        r.w[j] = read_tr8(st + boff[j]);
        r.s[j] = *reinterpret_cast<const u32x2*>(st + zoff + 32 * j + 8 * g4);
        r.z[j] = st[zoff + 64 + 16 * j + (lane & 15)];
      } else {
        r.w[2 * j] = read_tr8(st + boff[j]);
        r.w[2 * j + 1] = read_tr8(st + boff[j] + 32 * kQtCols);
      }
    }
  };
  // Dword c % 4 of bf[h][c / 4].
  auto convert = [&](const Raw& r, int h, int c) {
    const int j = c >> 2, d = c & 3;
    if constexpr (INT4) {
      const float z = (float)r.z[j];
      bf[h][j][d] = int4_pair(h ? r.w[j].y : r.w[j].x, d, -1024.f - z, -64.f - z);
    } else {
      bf[h][j][d] = int8_pair(r.w[2 * j + h], d);
    }
  };

  const int pre = NS < S ? NS : S;
  for (int t = 0; t < pre; ++t) {
#pragma unroll
    for (int u = 0; u < D; ++u) issue(sbase + (uint32_t)(t * STEP), u);
    advance();
  }
  if (NS >= S) vm_wait(D * (S - 1));
  else vm_wait(0);
  asm volatile("s_barrier" ::: "memory");
  read_raw(ring, raw);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < TM; ++i) read_a(ring, h, i);
#pragma unroll
  for (int c = 0; c < 4 * TN; ++c) convert(raw, 0, c);

  // One step: MFMAs of step t from registers; the slot of step t, whose
  // fragments every wave holds past the barrier, is filled with step t + S
  // (MORE); step t + 1 is read from LDS, and the conversions run between the
  // MFMAs, half a step ahead of their use.  (After the last step the reads
  // take a stale slot, unused.)
  int slot = 0;
  auto step = [&](auto more) {
    constexpr bool MORE = decltype(more)::value;
    const int slot_nx = slot + 1 == S ? 0 : slot + 1;
    const unsigned char* nx = ring + slot_nx * STEP;
    const uint32_t fill = sbase + (uint32_t)(slot * STEP);
    Raw r;
    read_raw(nx, r);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);  // (else every fragment is held twice)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = mfma16x16x32(bf[h][j], af[h][i], INT4 && h == 0 ? zero4 : acc[i][j]);
        read_a(nx, h, i);
#pragma unroll
        for (int c = i * 4 * TN / TM; c < (i + 1) * 4 * TN / TM; ++c) convert(h == 0 ? raw : r, 1 - h, c);
        if constexpr (MORE) {
#pragma unroll
          for (int u = (h * TM + i) * D / (2 * TM); u < (h * TM + i + 1) * D / (2 * TM); ++u) issue(fill, u);
        }
      }
    }
    if constexpr (MORE) advance();
    if constexpr (INT4) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const u32x2 sc = raw.s[j];  // the scales of this lane's four columns
        const float s4[4] = {bf16_to_f32(sc.x & 0xffffu), bf16_to_f32(sc.x >> 16), bf16_to_f32(sc.y & 0xffffu),
                             bf16_to_f32(sc.y >> 16)};
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) y[i][j][e] = __builtin_fmaf(s4[e], acc[i][j][e], y[i][j][e]);
      }
    }
    raw = r;
    slot = slot_nx;
  };
  // This wave's pieces of step t + 1 landed (n: steps after it in flight)
  // and its fragments in registers; past the barrier so are every wave's.
  auto sync = [&](int n) {
    __builtin_amdgcn_sched_barrier(0);
    vm_wait(n * D);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  int t = 0;
  for (; t + S < NS; ++t) {
    sync(S - 2);
    step(std::true_type{});
  }
  for (; t < NT; ++t) {
    switch (NS - 2 - t) {  // fewer than S - 1
      case 1: sync(1); break;
      case 2: sync(2 <= S - 2 ? 2 : 0); break;
      case 3: sync(3 <= S - 2 ? 3 : 0); break;
      case 4: sync(4 <= S - 2 ? 4 : 0); break;
      default: sync(0); break;
    }
    if (KW == 1 || t < NS) step(std::false_type{});
  }
  if constexpr (INT4) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = y[i][j];
  }

  // The wave groups' sums through LDS; each group then carries 1/KW of the
  // TM x TN blocks of the tile on, block kw * NB + u at b[u].
  constexpr int NB = TM * TN / KW;
  static_assert(NB * KW == TM * TN, "blocks divide over the wave groups");
  f32x4 b[NB];
  if constexpr (KW == 1) {
#pragma unroll
    for (int u = 0; u < NB; ++u) b[u] = acc[u / TN][u % TN];
  } else {
    __syncthreads();
    f32x4* const red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int u = 0; u < TM * TN; ++u) red[(kw * TM * TN + u) * 256 + tid] = acc[u / TN][u % TN];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      b[u] = red[(kw * NB + u) * 256 + tid];
#pragma unroll
      for (int q = 1; q < KW; ++q) b[u] += red[(q * TM * TN + kw * NB + u) * 256 + tid];
    }
  }

  if (p.ks > 1) {
    constexpr int PART = BM * kQtCols;
    float* tp = p.part + (int64_t)tile * p.ks * PART;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(tp, 0, p.ks * PART * 4, kBufWord3);
#pragma unroll
    for (int u = 0; u < NB; ++u)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, b[u]), rs,
                                             ((TM * TN * ksi + kw * NB + u) * 256 + tid) * 16, 0, kSc1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every partial store acknowledged
    __syncthreads();
    volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(smem);
    if (threadIdx.x == 0) {
      uint32_t* ctr = p.cnt + tile;
      asm volatile("" : "+v"(ctr));  // per-lane address: a vector atomic
      const uint32_t old = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t last = old == (uint32_t)(p.ks - 1);
      if (last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last;
    }
    __syncthreads();
    if (!*flag) return;
    // The partials in k order, this workgroup's from memory too.
#pragma unroll
    for (int u = 0; u < NB; ++u) b[u] = zero4;
    for (int q = 0; q < p.ks; ++q) {
#pragma unroll
      for (int u = 0; u < NB; ++u)
        b[u] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rs, ((TM * TN * q + kw * NB + u) * 256 + tid) * 16, 0, kSc1));
    }
  }

  // This lane holds row m, columns n .. n + 3 of each 16 x 16 block.
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int blk = kw * NB + u, i = blk / TN, j = blk % TN;
    const int n = n0w + 16 * j + 4 * g4, m = m0 + 16 * i + (lane & 15);
    if (n >= N || m >= M) continue;
    if constexpr (!INT4) b[u] *= *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.s) + n);
    epi_store_bf16x4(p.y, p.aux, p.epi, (size_t)m * N + n, b[u]);
  }
}

}  // namespace mk

namespace mkq {
namespace {

constexpr int64_t kCounterBytes = 64 * 1024;
constexpr int kCounters = 16384;
constexpr int kCus = 256;

template <bool INT4, int BM, int S, int KW>
hipError_t launch(const mk::QTileArgs& a, unsigned grid, hipStream_t st) {
  constexpr int ring = KW * S * (BM * 128 + (INT4 ? 32 * 128 + 1024 : 64 * 128)), red = KW * BM * mk::kQtCols * 4;
  constexpr int lds = ring > red ? ring : red;
  auto* fn = a.N % 16 == 0 ? mk::qtile_kernel<INT4, BM, S, KW, false> : mk::qtile_kernel<INT4, BM, S, KW, true>;
  const hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(256 * KW), lds, st, a);
  return hipGetLastError();
}

}  // namespace

// Cost model, us (17 to 2000 rows of K, N = 4096 x 14336, 4096 x 1792 and
// 1088 x 3008, within a tenth): 3 to launch; a round of 256 workgroups 1.2 +
// 0.02 BM to fill the ring and store, and 0.137 + 0.0021 BM (int8) or 0.225 +
// 0.00255 BM (int4) a 64-k step; a K split 3 + 0.35 ks and its partials at
// 9 MB a us.  K is split only into a grid of at most two rounds.
// MK_QMM_QT_BM / MK_QMM_QT_KS restrict the choice to one tile or split.
bool qtile_plan(bool int4, int64_t M, int64_t K, int64_t N, int64_t cap, QTilePlan* p) {
  if (K % 64 != 0 || N % 8 != 0 || M < 1 || K > (1 << 22) || N > (1 << 25)) return false;
  const char *bm_env = getenv("MK_QMM_QT_BM"), *ks_env = getenv("MK_QMM_QT_KS");
  const int64_t tiles_n = (N + mk::kQtCols - 1) / mk::kQtCols, groups = K / 64;
  bool have = false;
  for (int bm : {32, 64, 96, 128}) {
    if (bm_env && atoi(bm_env) != bm) continue;
    const int64_t tiles = ((M + bm - 1) / bm) * tiles_n;
    for (int ks : {1, 2, 3, 4, 6, 8}) {
      if (ks_env && atoi(ks_env) != ks) continue;
      if (ks > 1 && (groups < ks || tiles > kCounters)) break;
      if (ks > 1 && !ks_env && (groups < 4 * ks || tiles * ks > 2 * kCus)) break;
      const int64_t bytes = ks > 1 ? kCounterBytes + tiles * ks * bm * mk::kQtCols * 4 : 0;
      if (bytes > cap || tiles * ks > (1 << 24)) break;
      const double rounds = std::ceil((double)(tiles * ks) / kCus), steps = std::ceil((double)groups / ks);
      const double step = int4 ? 0.225 + 0.00255 * bm : 0.137 + 0.0021 * bm;
      const double us = 3.0 + rounds * (1.2 + 0.02 * bm + steps * step) + (ks > 1 ? 3.0 + 0.35 * ks + bytes / 9e6 : 0.0);
      if (!have || us < p->us) {
        *p = QTilePlan{bm, ks, bytes, us};
        have = true;
      }
    }
  }
  return have;
}

bool qtile_aligned(bool int4, const void* x, const void* w, const void* s, const void* z, const void* y,
                   const void* aux, int64_t N) {
  auto off = [](const void* q, unsigned a) { return (reinterpret_cast<uintptr_t>(q) & (a - 1)) != 0; };
  return !off(x, 16) && !off(w, N % 16 == 0 ? 16 : 4) && !off(s, int4 ? 4 : 16) && !(int4 && off(z, 4)) && !off(y, 8) &&
         !off(aux, 8);
}

hipError_t qtile_launch(bool int4, const void* x, const void* w, const void* s, const void* z, void* y, int64_t M,
                        int64_t K, int64_t N, const void* aux, int epi, const QTilePlan& p, void* workspace,
                        hipStream_t stream) {
  mk::QTileArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.w = static_cast<const uint8_t*>(w);
  a.s = s;
  a.z = static_cast<const uint8_t*>(z);
  a.y = static_cast<uint16_t*>(y);
  a.aux = static_cast<const uint16_t*>(aux);
  a.epi = epi;
  a.M = (int)M;
  a.K = (int)K;
  a.N = (int)N;
  a.ks = p.ks;
  a.cnt = p.ks > 1 ? static_cast<uint32_t*>(workspace) : nullptr;
  a.part = p.ks > 1 ? reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + kCounterBytes) : nullptr;
  const unsigned grid =
      (unsigned)(((M + p.bm - 1) / p.bm) * ((N + mk::kQtCols - 1) / mk::kQtCols) * p.ks);
  if (int4) {
    switch (p.bm) {
      case 32: return launch<true, 32, 4, 4>(a, grid, stream);
      case 64: return launch<true, 64, 6, 2>(a, grid, stream);
      case 96: return launch<true, 96, 4, 2>(a, grid, stream);
      default: return launch<true, 128, 3, 2>(a, grid, stream);
    }
  }
  switch (p.bm) {
    case 32: return launch<false, 32, 3, 4>(a, grid, stream);
    case 64: return launch<false, 64, 5, 2>(a, grid, stream);
    case 96: return launch<false, 96, 4, 2>(a, grid, stream);
    default: return launch<false, 128, 3, 2>(a, grid, stream);
  }
}

}  // namespace mkq
