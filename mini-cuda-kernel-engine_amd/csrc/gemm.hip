// gemm.hip -- launch_gemm_f32 and gemm_kernel_attrs for every GemmVariant.
//
// Replaces kernels/gemm.cu (launcher gemm.cu:829-882, dispatch table :595-700,
// attribute query :884-904).  The fast path is the appended kMfmaF32 variant
// (gemm_mfma.hpp).  The reference's FMA ladder is kept so that every variant a
// caller may name still runs and stays correct, re-shaped for wave64:
//   kNaive / kNaiveUncoalesced  one lane per output; 64 x 4 workgroups with lane x
//                               on the C column (coalesced) or on the C row;
//   kTiledSmem                  32 x 32 x 32 LDS tiles, one output per lane
//                               (tile (32,32,32,1,1), 1024 lanes);
//   kTiledRegBlock, kWarpTile,  128 x 128 block tile, BK = 8, 8 x 8 outputs per
//   kWarpTileNoDbuf,            lane, A staged transposed in LDS; the variants
//   kWarpTileVec4               differ in lane map (row-major vs 8 x 8 per wave64),
//                               LDS double buffering, and 16-byte global loads;
//   kCublasRef                  the vendor-library ceiling row (rocBLAS).
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "common.hpp"
#include "device_math.hpp"
#include "gemm_mfma.hpp"
#include "gemm_rows.hpp"

namespace mcke_amd {
namespace {

// ---------------------------------------------------------------------------
// Ladder kernels (CUDA-core-style FMA paths)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void store_c(float* c, float acc, float alpha, float beta) {
  *c = (beta == 0.0f) ? alpha * acc : alpha * acc + beta * *c;
}

template <bool COALESCED>
__global__ __launch_bounds__(256) void gemm_naive_kernel(const float* __restrict__ a,
                                                         const float* __restrict__ b,
                                                         float* __restrict__ c, int m, int n,
                                                         int k, float alpha, float beta) {
  const int col = COALESCED ? blockIdx.x * 64 + threadIdx.x : blockIdx.x * 4 + threadIdx.y;
  const int row = COALESCED ? blockIdx.y * 4 + threadIdx.y : blockIdx.y * 64 + threadIdx.x;
  if (row >= m || col >= n) return;
  float acc = 0.0f;
  for (int p = 0; p < k; ++p)
    acc += a[static_cast<int64_t>(row) * k + p] * b[static_cast<int64_t>(p) * n + col];
  store_c(c + static_cast<int64_t>(row) * n + col, acc, alpha, beta);
}

__global__ __launch_bounds__(1024) void gemm_tiled_smem_kernel(const float* __restrict__ a,
                                                               const float* __restrict__ b,
                                                               float* __restrict__ c, int m,
                                                               int n, int k, float alpha,
                                                               float beta) {
  constexpr int T = 32;
  __shared__ float As[T][T + 1];
  __shared__ float Bs[T][T];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int row = blockIdx.y * T + ty, col = blockIdx.x * T + tx;
  float acc = 0.0f;
  for (int kt = 0; kt < steps_along(k, T); ++kt) {
    const int k0 = kt * T;
    As[ty][tx] = (row < m && k0 + tx < k) ? a[static_cast<int64_t>(row) * k + k0 + tx] : 0.0f;
    Bs[ty][tx] = (k0 + ty < k && col < n) ? b[static_cast<int64_t>(k0 + ty) * n + col] : 0.0f;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < T; ++p) acc += As[ty][p] * Bs[p][tx];
    __syncthreads();
  }
  if (row < m && col < n) store_c(c + static_cast<int64_t>(row) * n + col, acc, alpha, beta);
}

// Register-blocked 128x128x8, 8x8 per lane, 256 lanes.
// LANE_MAP 0: lane t -> (ty, tx) = (t / 16, t % 16), row-major over the 16x16 grid.
// LANE_MAP 1: each wave64 owns an 8x8 patch of the lane grid (64 x 64 outputs), so a
//             wave reads 8 distinct A and 8 distinct B fragments from LDS per k.
template <int LANE_MAP, bool DBUF, int VW>
__global__ __launch_bounds__(256) void gemm_regblock_kernel(const float* __restrict__ a,
                                                            const float* __restrict__ b,
                                                            float* __restrict__ c, int m,
                                                            int n, int k, float alpha,
                                                            float beta) {
  constexpr int BM = 128, BN = 128, BK = 8, TM = 8, TN = 8;
  constexpr int APAD = 4;
  constexpr int NBUF = DBUF ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float As[NBUF][BK][BM + APAD];
  __shared__ __attribute__((aligned(16))) float Bs[NBUF][BK][BN];

  const int t = threadIdx.x;
  int ty, tx;
  if (LANE_MAP == 0) {
    ty = t / 16;
    tx = t % 16;
  } else {
    const int w = t / 64, l = t % 64;
    ty = (w / 2) * 8 + l / 8;
    tx = (w % 2) * 8 + l % 8;
  }
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

  // Global -> LDS mapping: A tile 128 x 8 (1024 floats), B tile 8 x 128 (1024 floats);
  // four floats per lane each, as one float4 (VW == 4) or four scalars.
  const int a_row = t / 2, a_col = (t % 2) * 4;      // A: 2 lanes per row of 8
  const int b_row = t / 32, b_col = (t % 32) * 4;    // B: 32 lanes per row of 128

  float ra[4], rb[4];
  auto gload = [&](int k0) {
    const int gm = m0 + a_row;
    if (VW == 4) {
      f32x4 va{0.f, 0.f, 0.f, 0.f}, vb{0.f, 0.f, 0.f, 0.f};
      if (gm < m && k0 + a_col < k)
        va = *reinterpret_cast<const f32x4*>(a + static_cast<int64_t>(gm) * k + k0 + a_col);
      if (k0 + b_row < k && n0 + b_col < n)
        vb = *reinterpret_cast<const f32x4*>(b + static_cast<int64_t>(k0 + b_row) * n + n0 + b_col);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ra[i] = va[i];
        rb[i] = vb[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gk = k0 + a_col + i;
        ra[i] = (gm < m && gk < k) ? a[static_cast<int64_t>(gm) * k + gk] : 0.0f;
        const int gn = n0 + b_col + i;
        rb[i] = (k0 + b_row < k && gn < n) ? b[static_cast<int64_t>(k0 + b_row) * n + gn] : 0.0f;
      }
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) As[buf][a_col + i][a_row] = ra[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) Bs[buf][b_row][b_col + i] = rb[i];
  };

  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.0f;

  auto compute = [&](int buf) {
#pragma unroll
    for (int p = 0; p < BK; ++p) {
      float av[TM], bv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) av[i] = As[buf][p][ty * TM + i];
#pragma unroll
      for (int j = 0; j < TN; ++j) bv[j] = Bs[buf][p][tx * TN + j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += av[i] * bv[j];
    }
  };

  const int ktiles = steps_along(k, BK);
  if (DBUF) {
    if (ktiles > 0) {
      gload(0);
      sstore(0);
    }
    __syncthreads();
    for (int kt = 0; kt < ktiles; ++kt) {
      const int cur = kt & 1;
      const bool more = kt + 1 < ktiles;
      if (more) gload((kt + 1) * BK);
      compute(cur);
      if (more) sstore(cur ^ 1);
      __syncthreads();
    }
  } else {
    for (int kt = 0; kt < ktiles; ++kt) {
      gload(kt * BK);
      sstore(0);
      __syncthreads();
      compute(0);
      __syncthreads();
    }
  }

#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = m0 + ty * TM + i;
    if (row >= m) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + tx * TN + j;
      if (col < n) store_c(c + static_cast<int64_t>(row) * n + col, acc[i][j], alpha, beta);
    }
  }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------
bool tile_eq(const mcke_gemm_tile& t, int bm, int bn, int bk, int tm, int tn) {
  return t.bm == bm && t.bn == bn && t.bk == bk && t.tm == tm && t.tn == tn;
}

// gemm_tile.hpp:112-124 with a 64-lane wavefront.
bool tile_self_consistent(const mcke_gemm_tile& t) {
  if (t.bm <= 0 || t.bn <= 0 || t.bk <= 0 || t.tm <= 0 || t.tn <= 0) return false;
  if (t.bm % t.tm != 0 || t.bn % t.tn != 0) return false;
  const int threads = (t.bm / t.tm) * (t.bn / t.tn);
  if (threads <= 0 || threads > 1024) return false;
  if (threads % kWave != 0) return false;
  if ((t.bm * t.bk) % threads != 0) return false;
  if ((t.bk * t.bn) % threads != 0) return false;
  return true;
}

// CUs of the current device (cached per device); 256, the gfx950 part's count,
// when no device can be queried (a CPU-only host asking for a tile).
int64_t device_cu_count() {
  static std::mutex mu;
  static std::vector<int> cached;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
    (void)hipGetLastError();
    return 256;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (static_cast<int>(cached.size()) <= dev) cached.resize(dev + 1, 0);
  if (cached[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0) {
      (void)hipGetLastError();
      cus = 256;
    }
    cached[dev] = cus;
  }
  return cached[dev];
}

using GemmFn = void (*)(const float*, const float*, float*, int, int, int, float, float);
using MfmaFn = void (*)(const float*, const float*, float*, int, int, int, float, float, int,
                        int, EpiArgs);

// MFMA instantiations: (bm, bn, bk) with tm = bm/16, tn = bn/16 (256 lanes).
// `even`: 16-byte path for M, N, K multiples of the tile (no bounds checks);
// `vec`: 16-byte path with bounds checks; `scalar`: any shape and alignment.
struct MfmaCfg {
  int bm, bn, bk;
  MfmaFn even, vec, scalar;
  int even_threads;   // block size of `even` (the staged kernels use 256)
  // `even` is the direct-to-LDS kernel, whose per-lane source offsets are 32-bit
  // byte offsets within a tile's BM rows of A and 32 rows of B.
  bool even_dma = false;
  // The same three kernels with the fused bias + activation epilogue.
  MfmaFn even_f = nullptr, vec_f = nullptr, scalar_f = nullptr;
  // The direct-to-LDS kernel's form for any M, N >= bn, K >= 32 and 4-byte alignment.
  MfmaFn edge = nullptr, edge_f = nullptr;
};

#define MCKE_MFMA_CFG(BM, BN, BK)                                                     \
  {BM, BN, BK, &gemm_mfma_kernel<BM, BN, BK, true, true>,                            \
   &gemm_mfma_kernel<BM, BN, BK, true, false>, &gemm_mfma_kernel<BM, BN, BK, false, false>, \
   kMfmaThreads, false, &gemm_mfma_kernel<BM, BN, BK, true, true, true>,             \
   &gemm_mfma_kernel<BM, BN, BK, true, false, true>,                                  \
   &gemm_mfma_kernel<BM, BN, BK, false, false, true>}
// BK = 32 whole tiles take the direct-to-LDS kernel (ST stages, KS wave groups
// splitting each stage's K range).
#define MCKE_MFMA_CFG_DMA(BM, BN, ST, KS)                                             \
  {BM, BN, 32, &gemm_mfma_dma_kernel<BM, BN, ST, KS>,                                \
   &gemm_mfma_kernel<BM, BN, 32, true, false>, &gemm_mfma_kernel<BM, BN, 32, false, false>, \
   kDmaThreads<BM, BN, KS>, true, &gemm_mfma_dma_kernel<BM, BN, ST, KS, true>,        \
   &gemm_mfma_kernel<BM, BN, 32, true, false, true>,                                  \
   &gemm_mfma_kernel<BM, BN, 32, false, false, true>,                                 \
   &gemm_mfma_dma_kernel<BM, BN, ST, KS, false, true>,                                \
   &gemm_mfma_dma_kernel<BM, BN, ST, KS, true, true>}

// 64 x 64 tiles serve small problems, whose single round of tiles leaves one
// workgroup per CU.  Their direct-to-LDS kernel meets at its barrier in the
// middle of a K step and keeps the fragment reads one sub-step ahead across it,
// so one wave group of 4 waves and a 4-stage ring measured best (1024^3: 109-110
// TFLOP/s vs 106-107 with two wave groups and 99-106 with the earlier 8-stage
// two-group ring; 2048^3 with 64 x 64 tiles: 134-135 vs 131; 3072^3: 136.5 vs
// 134; 3, 5, 6 and 8 stages all measured slower).  For 128 x 128 a 4-stage ring
// bought nothing over 2 at 2048^3 (137-139 either way).  32 x 32 tiles (one wave
// wide, four groups) give the smallest problems four times the workgroups of
// 64 x 64: 40.0 vs 22.6 TFLOP/s at 512^3, 7.0 vs 4.5 at 256^3.
const MfmaCfg kMfmaCfgs[] = {
    MCKE_MFMA_CFG_DMA(256, 256, 2, 1), MCKE_MFMA_CFG(256, 256, 16),
    MCKE_MFMA_CFG_DMA(128, 128, 2, 1), MCKE_MFMA_CFG(128, 128, 16),
    MCKE_MFMA_CFG_DMA(64, 64, 4, 1), MCKE_MFMA_CFG_DMA(32, 32, 4, 4),
};
#undef MCKE_MFMA_CFG
#undef MCKE_MFMA_CFG_DMA

// Direct-to-LDS kernels that a 64 x 64 launch runs where their tiles fill the CUs better
// (tile_us below): 128 x 64 at 144 against 138 TFLOP/s where there are tiles enough, and
// 32 x 64 (two wave groups over K) at 128 TFLOP/s where 64 x 64 tiles leave CUs with one
// against others' two.  Block sizes are all kMfmaThreads.
struct SubTile {
  int bm, bn;
  MfmaFn even, edge, even_f, edge_f;
};
#define MCKE_SUB(BM, BN, ST, KS)                                                       \
  {BM, BN, &gemm_mfma_dma_kernel<BM, BN, ST, KS, false, false>,                        \
   &gemm_mfma_dma_kernel<BM, BN, ST, KS, false, true>,                                 \
   &gemm_mfma_dma_kernel<BM, BN, ST, KS, true, false>,                                 \
   &gemm_mfma_dma_kernel<BM, BN, ST, KS, true, true>}
const SubTile kSubTiles64[] = {MCKE_SUB(128, 64, 2, 1), MCKE_SUB(32, 64, 4, 2)};
#undef MCKE_SUB
static_assert(kDmaThreads<128, 64, 1> == kMfmaThreads && kDmaThreads<32, 64, 2> == kMfmaThreads &&
                  kDmaThreads<64, 64, 1> == kMfmaThreads,
              "one block size");

// What a launch of bm x bn tiles takes, in us per 4096 of K: the time of its busiest CU,
// which runs r = ceil(tiles / CUs) of them, from launches timed on MI355X (gfx950, 256
// CUs) after 100 ms of warm-up.  K itself scales all alike, down to about 256; below that a
// tile's fixed cost shows (tile_fixed_us).
//   32 x 32:   26 alone on its CU, then 18.4 r (16 x 4096: 25.7; 480 x 816: 35 at r = 2;
//              1000 x 1024: 69 .. 73 at r = 4; 2602 x 1960: 364 .. 382 at r = 20).
//   32 x 64:   40 alone, then 34.5 r (1500 x 1000: 118 at r = 3; 1531 x 1021: 108 at r = 3;
//              2048 x 2048: 270 at r = 8; 4096 x 4096: 1077 at r = 32).
//   64 x 64:   69 alone, then 64.5 r (1024 x 1024: 67 .. 77; 1531 x 1021: 128 at r = 2;
//              1000 x 4096: 261 at r = 4; 3000 x 4096: 762 at r = 12).
//   128 x 64:  130 alone, then 10 + 122 r (1000 x 4096: 258 at r = 2; 2000 x 3000: 387 at
//              r = 3; 3000 x 4096: 732 at r = 6; 4096 x 4096: 954 at r = 8).
//   128 x 128: 257 alone, then 240 r, two tiles at a time: an odd last one shares its CU
//              with nothing, or falls to a CU that has two (r = 3: 755 .. 949, so r + 0.6).
//              2048 x 2048: 247 .. 269, 2048 x 4096: 511, 4096 x 4096: 937 .. 956.
//   256 x 256: 950 r, one at a time (4096 x 4096: 926 .. 974).
double tile_us(int bm, int bn, int64_t m, int64_t n, int64_t cus) {
  const int64_t tiles = ((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  const double r = static_cast<double>(tiles > cus ? (tiles + cus - 1) / cus : 1);
  const bool alone = tiles <= cus;
  switch (bm * bn) {
    case 32 * 32: return alone ? 26.0 : 18.4 * r;
    case 32 * 64: return alone ? 40.0 : 34.5 * r;
    case 64 * 64: return alone ? 69.0 : 64.5 * r;
    case 128 * 64: return alone ? 130.0 : 10.0 + 122.0 * r;
    case 128 * 128:
      return alone ? 257.0 : 240.0 * (r + (static_cast<int64_t>(r) % 2 == 1 ? 0.6 : 0.0));
    default: return 950.0 * r;
  }
}

// What a tile costs whatever its K: its prologue and its C store.  Fitted to launches of K 4
// to 256 over 75 shapes (us: 32 x 32 0.45 .. 0.57 a tile, 32 x 64 0.44, 64 x 64 0.6 .. 1.4,
// 128 x 128 2.1 .. 5).  Without it the smallest tile was taken for them: 576 x 3904 x 48
// 11.2 us at 32 x 32 against 8.6 at 64 x 64, 4614 x 6836 x 16 52.4 at 128 x 128 against 46.9.
double tile_fixed_us(int bm, int bn, int64_t m, int64_t n, int64_t cus) {
  const int64_t tiles = ((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  const double r = static_cast<double>((tiles + cus - 1) / cus);
  switch (bm * bn) {
    case 32 * 32: return 0.4 * r;
    case 32 * 64: return 0.5 * r;
    case 64 * 64: return 0.8 * r;
    case 128 * 128: return 4.0 * r;
    default: return 16.0 * r;   // 256 x 256
  }
}

const MfmaCfg* find_mfma(const mcke_gemm_tile& t) {
  for (const MfmaCfg& c : kMfmaCfgs)
    if (tile_eq(t, c.bm, c.bn, c.bk, c.bm / 16, c.bn / 16)) return &c;
  return nullptr;
}

struct Spec {
  const void* kernel = nullptr;   // for attribute queries
  GemmFn fn = nullptr;
  MfmaFn mfma = nullptr;
  MfmaFn mfma_even = nullptr;     // unchecked 16-byte variant for whole tiles
  MfmaFn mfma_f = nullptr;        // the two with the fused bias + activation epilogue
  MfmaFn mfma_even_f = nullptr;
  MfmaFn mfma_edge = nullptr;     // direct-to-LDS kernel for shapes that are not whole tiles
  MfmaFn mfma_edge_f = nullptr;
  int even_threads = 0;           // their block size
  bool even_dma = false;          // they take 32-bit per-lane source offsets
  dim3 block{1, 1, 1};
  int threads = 0;                // block size of `kernel`
  int tile_m = 0, tile_n = 0, tile_k = 0;
};

int gemm_spec(int variant, const mcke_gemm_tile* tile, bool vec4, Spec& s) {
  switch (variant) {
    case MCKE_GEMM_NAIVE:
      s.fn = &gemm_naive_kernel<true>;
      s.block = dim3(64, 4, 1);
      s.threads = 256;
      s.tile_m = 4;
      s.tile_n = 64;
      break;
    case MCKE_GEMM_NAIVE_UNCOALESCED:
      s.fn = &gemm_naive_kernel<false>;
      s.block = dim3(64, 4, 1);
      s.threads = 256;
      s.tile_m = 64;
      s.tile_n = 4;
      break;
    case MCKE_GEMM_TILED_SMEM:
      if (!tile || !tile_self_consistent(*tile))
        return invalid("launch_gemm_f32: tile is not self-consistent");
      if (!tile_eq(*tile, 32, 32, 32, 1, 1))
        return invalid("launch_gemm_f32: kTiledSmem is only instantiated for tile "
                       "(bm,bn,bk,tm,tn) = (32,32,32,1,1); no fallback is applied");
      s.fn = &gemm_tiled_smem_kernel;
      s.block = dim3(32, 32, 1);
      s.threads = 1024;
      s.tile_m = s.tile_n = 32;
      break;
    case MCKE_GEMM_TILED_REGBLOCK:
    case MCKE_GEMM_WARP_TILE:
    case MCKE_GEMM_WARP_TILE_NODBUF:
    case MCKE_GEMM_WARP_TILE_VEC4:
      if (!tile || !tile_self_consistent(*tile))
        return invalid("launch_gemm_f32: tile is not self-consistent");
      if (!tile_eq(*tile, 128, 128, 8, 8, 8))
        return invalid("launch_gemm_f32: the register-blocked variants are only instantiated "
                       "for tile (bm,bn,bk,tm,tn) = (128,128,8,8,8); no fallback is applied");
      if (variant == MCKE_GEMM_TILED_REGBLOCK) s.fn = &gemm_regblock_kernel<0, false, 1>;
      else if (variant == MCKE_GEMM_WARP_TILE_NODBUF) s.fn = &gemm_regblock_kernel<1, false, 1>;
      else if (variant == MCKE_GEMM_WARP_TILE) s.fn = &gemm_regblock_kernel<1, true, 1>;
      else s.fn = vec4 ? &gemm_regblock_kernel<1, true, 4> : &gemm_regblock_kernel<1, true, 1>;
      s.block = dim3(256, 1, 1);
      s.threads = 256;
      s.tile_m = s.tile_n = 128;
      break;
    case MCKE_GEMM_MFMA_F32: {
      if (!tile || !tile_self_consistent(*tile))
        return invalid("launch_gemm_f32: tile is not self-consistent");
      const MfmaCfg* cfg = find_mfma(*tile);
      if (!cfg)
        return invalid("launch_gemm_f32: kMfmaF32 is instantiated for tiles (256,256,32,16,16), "
                       "(256,256,16,16,16), (128,128,32,8,8), (128,128,16,8,8), "
                       "(64,64,32,4,4) and (32,32,32,2,2); no fallback is applied");
      s.mfma = vec4 ? cfg->vec : cfg->scalar;
      s.mfma_even = vec4 ? cfg->even : nullptr;
      s.mfma_f = vec4 ? cfg->vec_f : cfg->scalar_f;
      s.mfma_even_f = vec4 ? cfg->even_f : nullptr;
      s.mfma_edge = cfg->edge;
      s.mfma_edge_f = cfg->edge_f;
      s.even_threads = cfg->even_threads;
      s.even_dma = cfg->even_dma;
      s.tile_k = cfg->bk;
      s.block = dim3(kMfmaThreads, 1, 1);
      s.threads = s.mfma_even ? cfg->even_threads : kMfmaThreads;
      s.tile_m = cfg->bm;
      s.tile_n = cfg->bn;
      break;
    }
    case MCKE_GEMM_CUBLAS_REF:
      return invalid("gemm_spec: the library ceiling row has no kernel of this library");
    default:
      return invalid("launch_gemm_f32: unknown GemmVariant " + std::to_string(variant));
  }
  // Attribute queries report the instantiation that whole-tile shapes run.
  s.kernel = s.fn ? reinterpret_cast<const void*>(s.fn)
                  : reinterpret_cast<const void*>(s.mfma_even ? s.mfma_even : s.mfma);
  return ok();
}

// ---------------------------------------------------------------------------
// kCublasRef: rocBLAS sgemm as the ceiling row.  Row-major C = A B is the
// column-major C^T = B^T A^T, i.e. a no-transpose sgemm with the operands swapped.
// One handle per stream, created on first use and kept for the process lifetime.
// ---------------------------------------------------------------------------
int rocblas_for_stream(hipStream_t s, rocblas_handle* out) {
  static std::mutex mu;
  static std::vector<std::pair<hipStream_t, rocblas_handle>> cache;
  std::lock_guard<std::mutex> lk(mu);
  for (const auto& kv : cache)
    if (kv.first == s) {
      *out = kv.second;
      return ok();
    }
  rocblas_handle h = nullptr;
  if (rocblas_create_handle(&h) != rocblas_status_success)
    return fail(MCKE_STATUS_DEVICE_ERROR, "rocblas_create_handle failed");
  if (rocblas_set_stream(h, s) != rocblas_status_success)
    return fail(MCKE_STATUS_DEVICE_ERROR, "rocblas_set_stream failed");
  cache.emplace_back(s, h);
  *out = h;
  return ok();
}

int launch_rocblas(const float* a, const float* b, float* c, int m, int n, int k, float alpha,
                   float beta, hipStream_t s) {
  rocblas_handle h = nullptr;
  if (int rc = rocblas_for_stream(s, &h)) return rc;
  const rocblas_status st = rocblas_sgemm(h, rocblas_operation_none, rocblas_operation_none,
                                          n, m, k, &alpha, b, n, a, k, &beta, c, n);
  if (st != rocblas_status_success)
    return fail(MCKE_STATUS_DEVICE_ERROR,
                std::string("rocblas_sgemm failed: ") + rocblas_status_to_string(st));
  return ok();
}

using RowsFn = void (*)(const float*, const float*, float*, int, int, int, float, float, int, int,
                        EpiArgs);

// The few-tiles kernel for a 32 x 32 tile launch, if it is the better one: the smallest of
// its tiles (16 x 16, 16 x 32, 32 x 32, and 16 x 64 for up to 16 rows) whose workgroups
// are all resident at once, one per CU.  More than that is slower (300 x 217 x 4072: 266
// tiles of 16 x 16 27.1 us, 133 of 16 x 32 19.3).  The wider ones need some K to pay for
// their sums: 16 x 32 ties at 7 x 6015 x 628 (7.4 us against 7.3 for the 32 x 32 tile) and
// leads at 128 x 1012 x 320 (4.4 against 4.5); 32 x 32 leads from K = 1024 on (512 x 512 x
// 1024: 7.7 against 8.7; 500 x 500 x 1000: 9.9 against 9.6); 16 x 64 trails at 16 x 16384 x
// 256 (6.1 against 5.6) and leads at 16 x 16384 x 4096.  K of 32 or less is one chunk, which
// one of the eight waves works on: the 32 x 32 tile leads there by 0.1 .. 0.3 of 4.3 us.
// Per-lane source offsets are 32-bit.
struct RowsPick {
  RowsFn fn = nullptr;
  int tiles_m = 0, tiles_n = 0;
};

RowsPick find_rows(int64_t m, int64_t n, int64_t k, bool fused) {
  RowsPick p;
  if (64 * k >= (int64_t{1} << 30) || 64 * n >= (int64_t{1} << 30)) return p;
  const int64_t cus = device_cu_count();
  auto fits = [&](int mt, int nw, int64_t min_k) {
    const int64_t tm = (m + 16 * mt - 1) / (16 * mt), tn = (n + 16 * nw - 1) / (16 * nw);
    p.tiles_m = static_cast<int>(tm);
    p.tiles_n = static_cast<int>(tn);
    return n >= 16 * nw && k >= min_k && tm * tn <= cus;
  };
#define MCKE_ROWS(MT, NW, MIN_K)                                                              \
  if (fits(MT, NW, MIN_K)) {                                                                  \
    p.fn = fused ? &gemm_rows_kernel<MT, NW, true> : &gemm_rows_kernel<MT, NW, false>;        \
    return p;                                                                                 \
  }
  MCKE_ROWS(1, 1, 33)
  MCKE_ROWS(1, 2, 320)
  MCKE_ROWS(2, 2, 1024)
  if (m <= 16) MCKE_ROWS(1, 4, 1024)
#undef MCKE_ROWS
  return p;
}

// The register-staged kernel at the requested tile: any shape and alignment.
int launch_mfma_staged(const char* who, const Spec& sp, bool fused, const float* a, const float* b,
                       float* c, int64_t m, int64_t n, int64_t k, float alpha, float beta,
                       EpiArgs epi, hipStream_t s) {
  const int64_t tiles_m = (m + sp.tile_m - 1) / sp.tile_m;
  const int64_t tiles_n = (n + sp.tile_n - 1) / sp.tile_n;
  if (tiles_m * tiles_n > 2147483647LL)
    return invalid(std::string(who) + ": too many tiles for one launch");
  if (tiles_m * tiles_n * static_cast<int64_t>(sp.block.x) > int64_t{UINT32_MAX})
    return invalid(std::string(who) + ": tiles x lanes exceed the grid's 32-bit work size; use a "
                   "larger tile");
  MfmaFn fn = fused ? sp.mfma_f : sp.mfma;
  fn<<<static_cast<unsigned>(tiles_m * tiles_n), sp.block, 0, s>>>(
      a, b, c, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), alpha, beta,
      static_cast<int>(tiles_m), static_cast<int>(tiles_n), epi);
  MCKE_LAUNCH_CHECK(fused ? "gemm_mfma_kernel (bias + activation)" : "gemm_mfma_kernel");
  return ok();
}

// One kMfmaF32 launch: few tiles of 32 x 32 take the few-tiles kernel, whole tiles
// the direct-to-LDS kernel, and other shapes its EDGE form where a tile's columns fit in a
// row of B and K is long enough, else the staged kernel; `fused` picks the instantiations
// with the bias + activation epilogue, which route shapes exactly as the plain ones do
// (so a fused launch accumulates in the plain launch's order).
int launch_mfma(const char* who, const Spec& sp, bool fused, const float* a, const float* b,
                float* c, int64_t m, int64_t n, int64_t k, float alpha, float beta, EpiArgs epi,
                hipStream_t s) {
  // The kernels below load and store floats at 4-byte addresses.
  const bool floats = aligned(a, 4) && aligned(b, 4) && aligned(c, 4) && aligned(epi.bias, 4);
  if (sp.tile_m == 32 && floats && k > 0) {
    const RowsPick p = find_rows(m, n, k, fused);
    if (p.fn) {
      p.fn<<<static_cast<unsigned>(p.tiles_m * p.tiles_n), kRowsThreads, 0, s>>>(
          a, b, c, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), alpha, beta,
          p.tiles_m, p.tiles_n, epi);
      MCKE_LAUNCH_CHECK(fused ? "gemm_rows_kernel (bias + activation)" : "gemm_rows_kernel");
      return ok();
    }
  }
  int bm = sp.tile_m, bn = sp.tile_n;
  MfmaFn even = fused ? sp.mfma_even_f : sp.mfma_even;
  MfmaFn edge = fused ? sp.mfma_edge_f : sp.mfma_edge;
  // EDGE from K = 64 on.  Below that most of K is the remainder, and the staged kernel is as
  // fast or faster: 576 x 3904 x 40 8.5 us against 9.5, 4256 x 4864 x 40 40.1 against 46.8 at
  // 64 x 64, 4416 x 288 x 32 unaligned 6.2 against 6.7 at 32 x 32.  Only where it loads 4 bytes
  // at a time (`even` is null) do larger tiles gain from K = 32 on: 4614 x 6836 x 40 67 against 56.
  const bool edge_k = k >= (bm >= 64 && !even ? 32 : 64);
  if (bm == 64 && edge && floats && n >= 64 && (edge_k || (even && k == 32))) {
    const int64_t cus = device_cu_count();
    double best = tile_us(64, 64, m, n, cus);
    for (const SubTile& t : kSubTiles64) {
      const double us = tile_us(t.bm, t.bn, m, n, cus);
      if (us >= best || t.bm * k >= (int64_t{1} << 30)) continue;
      if (!edge_k && (m % t.bm != 0 || n % t.bn != 0)) continue;
      best = us;
      bm = t.bm;
      bn = t.bn;
      even = !even ? nullptr : fused ? t.even_f : t.even;
      edge = fused ? t.edge_f : t.edge;
    }
  }
  const int64_t tiles_m = (m + bm - 1) / bm;
  const int64_t tiles_n = (n + bn - 1) / bn;
  if (tiles_m * tiles_n > 2147483647LL)
    return invalid(std::string(who) + ": too many tiles for one launch");
  const bool offsets32 = static_cast<int64_t>(bm) * k < (int64_t{1} << 30) &&
                         static_cast<int64_t>(32) * n < (int64_t{1} << 30);
  const bool whole = even && m % bm == 0 && n % bn == 0 && k % sp.tile_k == 0 &&
                     (!sp.even_dma || offsets32);
  const bool ragged = !whole && edge && edge_k && n >= bn && offsets32 && floats;
  if (!whole && !ragged)
    return launch_mfma_staged(who, sp, fused, a, b, c, m, n, k, alpha, beta, epi, s);
  MfmaFn fn = whole ? even : edge;
  const dim3 block(static_cast<unsigned>(sp.even_threads), 1, 1);
  if (tiles_m * tiles_n * static_cast<int64_t>(block.x) > int64_t{UINT32_MAX})
    return invalid(std::string(who) + ": tiles x lanes exceed the grid's 32-bit work size; use a "
                   "larger tile");
  fn<<<static_cast<unsigned>(tiles_m * tiles_n), block, 0, s>>>(
      a, b, c, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), alpha, beta,
      static_cast<int>(tiles_m), static_cast<int>(tiles_n), epi);
  MCKE_LAUNCH_CHECK(fused ? "gemm_mfma_kernel (bias + activation)" : "gemm_mfma_kernel");
  return ok();
}

}  // namespace
}  // namespace mcke_amd

using namespace mcke_amd;

extern "C" {

int mcke_launch_gemm_f32(const float* a, const float* b, float* c, int64_t m, int64_t n,
                         int64_t k, float alpha, float beta, int variant,
                         const mcke_gemm_tile* tile, void* stream) {
  if (m == 0 || n == 0) return ok();
  if (m < 0 || n < 0 || k < 0) return invalid("launch_gemm_f32: negative extent");
  if (!a || !b || !c) return invalid("launch_gemm_f32: null pointer");
  if (a == c || b == c)
    return invalid("launch_gemm_f32: output aliases an input, which violates the "
                   "__restrict__ contract");
  if (m > 2147483647LL || n > 2147483647LL || k > 2147483647LL)
    return invalid("launch_gemm_f32: extent exceeds INT32_MAX");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = static_cast<int>(m), ni = static_cast<int>(n), ki = static_cast<int>(k);

  if (variant == MCKE_GEMM_CUBLAS_REF) return launch_rocblas(a, b, c, mi, ni, ki, alpha, beta, s);

  // 16-byte loads need every row start of A and B aligned: k % 4, n % 4 and the
  // base pointers (m is unconstrained).
  const bool vec4 = (k % 4 == 0) && (n % 4 == 0) && aligned(a, 16) && aligned(b, 16) &&
                    aligned(c, 16);
  Spec sp;
  if (int rc = gemm_spec(variant, tile, vec4, sp)) return rc;

  if (sp.mfma)
    return launch_mfma("launch_gemm_f32", sp, false, a, b, c, m, n, k, alpha, beta,
                       EpiArgs{nullptr, 0}, s);

  // grid.x walks C column tiles and grid.y C row tiles for every ladder kernel
  // (kNaiveUncoalesced only changes which lane index runs along a row).
  const int64_t gx = (n + sp.tile_n - 1) / sp.tile_n;
  const int64_t gy = (m + sp.tile_m - 1) / sp.tile_m;
  if (gy > 65535) return invalid("launch_gemm_f32: m too large for the grid's y limit");
  if (gx * static_cast<int64_t>(sp.block.x) > int64_t{UINT32_MAX})
    return invalid("launch_gemm_f32: n too large for the grid's 32-bit work size");
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy), 1);
  sp.fn<<<grid, sp.block, 0, s>>>(a, b, c, mi, ni, ki, alpha, beta);
  MCKE_LAUNCH_CHECK("gemm kernel");
  return ok();
}

int mcke_launch_gemm_bias_act_f32(const float* a, const float* b, const float* bias, float* y,
                                  int64_t m, int64_t n, int64_t k, float alpha, int activation,
                                  const mcke_gemm_tile* tile, void* stream) {
  if (m == 0 || n == 0) return ok();
  if (m < 0 || n < 0 || k < 0) return invalid("launch_gemm_bias_act_f32: negative extent");
  if (!a || !b || !bias || !y) return invalid("launch_gemm_bias_act_f32: null pointer");
  if (y == a || y == b || y == bias)
    return invalid("launch_gemm_bias_act_f32: the output aliases an input, which violates the "
                   "__restrict__ contract");
  if (activation < MCKE_ACT_NONE || activation > MCKE_ACT_GELU_TANH)
    return invalid("launch_gemm_bias_act_f32: unknown Activation " + std::to_string(activation));
  if (m > 2147483647LL || n > 2147483647LL || k > 2147483647LL)
    return invalid("launch_gemm_bias_act_f32: extent exceeds INT32_MAX");
  const bool vec4 = (k % 4 == 0) && (n % 4 == 0) && aligned(a, 16) && aligned(b, 16) &&
                    aligned(y, 16);
  Spec sp;
  if (int rc = gemm_spec(MCKE_GEMM_MFMA_F32, tile, vec4, sp)) return rc;
  return launch_mfma("launch_gemm_bias_act_f32", sp, true, a, b, y, m, n, k, alpha, 0.0f,
                     EpiArgs{bias, activation}, static_cast<hipStream_t>(stream));
}

int mcke_gemm_kernel_attrs(int variant, const mcke_gemm_tile* tile, mcke_kernel_attrs* out) {
  if (!out) return invalid("gemm_kernel_attrs: null out");
  if (variant == MCKE_GEMM_CUBLAS_REF)
    return fail(MCKE_STATUS_UNIMPLEMENTED,
                "gemm_kernel_attrs: the library ceiling row's kernels are not ours to introspect");
  Spec sp;
  if (int rc = gemm_spec(variant, tile, true, sp)) return rc;
  hipFuncAttributes fa{};
  MCKE_HIP_TRY(hipFuncGetAttributes(&fa, sp.kernel));
  out->regs_per_thread = fa.numRegs;
  out->agprs_per_thread = 0;   // not reported by the HIP runtime
  out->static_smem_bytes = fa.sharedSizeBytes;
  out->local_bytes = fa.localSizeBytes;
  out->threads_per_block = sp.threads;
  int blocks = 0;
  MCKE_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, sp.kernel, sp.threads, 0));
  out->max_blocks_per_sm_api = blocks;
  return ok();
}

int mcke_launch_gemm_lp_vendor(const void* a, const void* b, void* c, int ab_dtype,
                               int c_dtype, int64_t m, int64_t n, int64_t k, float alpha,
                               float beta, void* stream) {
  if ((ab_dtype != MCKE_DTYPE_BF16 && ab_dtype != MCKE_DTYPE_F16) ||
      (c_dtype != MCKE_DTYPE_F32 && c_dtype != ab_dtype))
    return invalid("launch_gemm_lp_vendor: (ab_dtype, c_dtype) must be (BF16|F16, F32|ab_dtype)");
  if (m == 0 || n == 0) return ok();
  if (m < 0 || n < 0 || k < 0) return invalid("launch_gemm_lp_vendor: negative extent");
  if (!a || !b || !c) return invalid("launch_gemm_lp_vendor: null pointer");
  if (a == c || b == c) return invalid("launch_gemm_lp_vendor: output aliases an input");
  if (m > 2147483647LL || n > 2147483647LL || k > 2147483647LL)
    return invalid("launch_gemm_lp_vendor: extent exceeds INT32_MAX");
  rocblas_handle h = nullptr;
  if (int rc = rocblas_for_stream(static_cast<hipStream_t>(stream), &h)) return rc;
  const rocblas_datatype ab =
      ab_dtype == MCKE_DTYPE_BF16 ? rocblas_datatype_bf16_r : rocblas_datatype_f16_r;
  const rocblas_datatype cd = c_dtype == MCKE_DTYPE_F32 ? rocblas_datatype_f32_r : ab;
  const int mi = static_cast<int>(m), ni = static_cast<int>(n), ki = static_cast<int>(k);
  // Row-major C = A B is the column-major C^T = B^T A^T: operands swapped.
  const rocblas_status st = rocblas_gemm_ex(
      h, rocblas_operation_none, rocblas_operation_none, ni, mi, ki, &alpha, b, ab, ni, a, ab, ki,
      &beta, c, cd, ni, c, cd, ni, rocblas_datatype_f32_r, rocblas_gemm_algo_standard, 0, 0);
  if (st != rocblas_status_success)
    return fail(MCKE_STATUS_DEVICE_ERROR,
                std::string("rocblas_gemm_ex failed: ") + rocblas_status_to_string(st));
  return ok();
}

int mcke_gemm_mfma_default_tile(int64_t m, int64_t n, int64_t k, mcke_gemm_tile* out) {
  if (!out) return invalid("gemm_mfma_default_tile: null out");
  // The tile whose launch is the shortest (tile_us, scaled to K up to 256 and with the tiles'
  // fixed cost), ties to the larger one; the 64 x 64 tile counts as the better of its own and
  // the 32 x 64 one that it may run where N and K are 64 or more.  Shapes that are not whole
  // tiles cost the two large tiles 3% more (the EDGE form's row and column checks: 1000 x 4096
  // x 1024 69.8 us against 68.0 for 1024 rows at 128 x 128).
  static const mcke_gemm_tile cands[] = {
      {256, 256, 32, 16, 16}, {128, 128, 32, 8, 8}, {64, 64, 32, 4, 4}, {32, 32, 32, 2, 2}};
  const int64_t cus = device_cu_count();
  auto launch_us = [&](int bm, int bn) {
    const double us = tile_us(bm, bn, m, n, cus);
    if (k > 256) return us;
    return us * static_cast<double>(k) / 4096.0 + tile_fixed_us(bm, bn, m, n, cus);
  };
  double best = 0.0;
  for (const mcke_gemm_tile& c : cands) {
    double us = launch_us(c.bm, c.bn);
    if (c.bm == 64 && n >= 64 && k >= 64) us = std::min(us, launch_us(32, 64));
    if (c.bm >= 128 && (m % c.bm != 0 || n % c.bn != 0 || k % 32 != 0)) us *= 1.03;
    if (c.bm == 256 || us < best) {
      best = us;
      *out = c;
    }
  }
  return ok();
}

}  // extern "C"
