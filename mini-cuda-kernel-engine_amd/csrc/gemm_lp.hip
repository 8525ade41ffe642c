// gemm_lp.hip -- the 16-bit-input GEMM entry points (bf16 / fp16 in, fp32
// accumulation, fp32 or 16-bit out) over gemm_lp.hpp.
//
// The reference reserves DType::kF16 and kBF16 (include/mcke/core/dtype.hpp:33-41)
// for tensor-core inputs but ships only the fp32 launcher (kernels.hpp:265-269,
// gemm.cu:829-882).  mcke_launch_gemm_lp keeps that launcher's argument order,
// validation and status codes, with the two dtypes added after the pointers.
#include <hip/hip_runtime.h>

#include <string>

#include "common.hpp"
#include "gemm_lp.hpp"
#include "gemm_lp_split.hpp"

namespace mcke_amd {
namespace {

using LpKernel = const void*;

// Direct-to-LDS 16x16x32 kernel for a BM x BN tile: whole tiles with 16-byte aligned
// operands and K % 64 == 0, or the EDGE form.  Its per-lane source offsets are 32-bit: BM
// rows of A and 64 rows of B must span less than 4 GiB.
template <int BM, int BN>
bool dma_offsets32(int n, int k) {
  return static_cast<int64_t>(BM) * k * 2 + 4096 < (int64_t{1} << 32) &&
         static_cast<int64_t>(64) * n * 2 < (int64_t{1} << 32);
}

int64_t tile_count(int m, int n, int bm, int bn) {
  return static_cast<int64_t>(steps_along(m, bm)) * steps_along(n, bn);
}

struct LpArgs {
  const uint16_t* a;
  const uint16_t* b;
  void* c;
  int m, n, k;
  float alpha, beta;
  hipStream_t s;
};

int check_grid(int64_t tiles, int threads) {
  if (tiles * threads > int64_t{UINT32_MAX})
    return invalid("launch_gemm_lp: tiles x lanes exceed the grid's 32-bit work size; use a "
                   "larger tile");
  return ok();
}

template <typename T, typename OutT, int BM, int BN, bool EDGE>
int launch_dma(const LpArgs& x) {
  const int64_t tiles = tile_count(x.m, x.n, BM, BN);
  if (int rc = check_grid(tiles, kMfmaThreads)) return rc;
  gemm_lp_dma16_kernel<T, OutT, BM, BN, EDGE>
      <<<static_cast<unsigned>(tiles), kMfmaThreads, 0, x.s>>>(
          x.a, x.b, static_cast<OutT*>(x.c), x.m, x.n, x.k, x.alpha, x.beta,
          steps_along(x.m, BM), steps_along(x.n, BN));
  MCKE_LAUNCH_CHECK("gemm_lp_dma16_kernel");
  return ok();
}

template <typename T, typename OutT, int MT, int NW, int WV>
int launch_split_as(const LpArgs& x) {
  constexpr int TM = 16 * MT, TN = 16 * NW;
  const int64_t tiles = tile_count(x.m, x.n, TM, TN);
  if (int rc = check_grid(tiles, WV * kWave)) return rc;
  gemm_lp_split_kernel<T, OutT, MT, NW, WV>
      <<<static_cast<unsigned>(tiles), WV * kWave, 0, x.s>>>(
          x.a, x.b, static_cast<OutT*>(x.c), x.m, x.n, x.k, x.alpha, x.beta,
          steps_along(x.m, TM), steps_along(x.n, TN));
  MCKE_LAUNCH_CHECK("gemm_lp_split_kernel");
  return ok();
}

// The split-K kernel by shape.  Few rows over up to 8192 columns: 32 columns a workgroup
// and 8 waves, for as many workgroups as there are (16 x 4096 x 4096: 16 x 32 11.9 us,
// 32 x 64 14.8, 64 x 64 16.4; 16 x 16384 x 4096: 38.6, 25.8, 26.8).  Else 32 x 64 up to
// four tiles per CU (64 x 4096 x 4096: 15.6 us against 21.3 for 64 x 64; 1628 x 800 x 1109:
// 14.9 against 17.4), 64 x 64 past that (1531 x 4096 x 1024: 28.2 against 33.3;
// 4032 x 843 x 2744: 62.7 against 83.8).  Widths of 32 .. 63 take 32 columns.
template <typename T, typename OutT>
int launch_split(const LpArgs& x) {
  if (x.n < 64 || (x.m <= 32 && x.n <= 8192))
    return x.m <= 16 ? launch_split_as<T, OutT, 1, 2, 8>(x) : launch_split_as<T, OutT, 2, 2, 8>(x);
  if (tile_count(x.m, x.n, 32, 64) <= 1024) return launch_split_as<T, OutT, 2, 4, 4>(x);
  return launch_split_as<T, OutT, 4, 4, 4>(x);
}

// The register-staged kernel's checked forms at the requested tile: what is narrower than
// any other kernel's tile, or past their 32-bit offsets or grids.
template <typename T, typename OutT, int BM, int BN>
int launch_staged(const LpArgs& x, bool vec) {
  const int64_t tiles = tile_count(x.m, x.n, BM, BN);
  if (int rc = check_grid(tiles, kMfmaThreads)) return rc;
  auto* fn = vec ? &gemm_lp_kernel<T, OutT, BM, BN, true, false>
                 : &gemm_lp_kernel<T, OutT, BM, BN, false, false>;
  fn<<<static_cast<unsigned>(tiles), kMfmaThreads, 0, x.s>>>(
      x.a, x.b, static_cast<OutT*>(x.c), x.m, x.n, x.k, x.alpha, x.beta,
      steps_along(x.m, BM), steps_along(x.n, BN));
  MCKE_LAUNCH_CHECK("gemm_lp_kernel");
  return ok();
}

// Short K over many tiles: the product is its C store, and the register-staged kernel's four
// waves share a tile's one stage where the split-K kernel has one wave work and three add
// zeros.  16-byte operands up to 63 of K (fp16 to fp16, 2460 x 1608 x 40: 6.7 us at 64 x 64
// against 9.9 for split K; up to 1024 tiles they tie, fp32 C, 853 x 1880 x 64 5.5 against 5.4),
// others up to 7, as their loads are element by element (fp32 C, 2293 x 1737 x 7: 10.3 against
// 12.8; x 15: 11.6 against 11.7).  128 x 128 tiles where they fill two rounds of CUs or more to 80%
// (2166 x 3544 x 40: 10.9 us against 12.1 at 64 x 64; 2460 x 1608, 260 tiles: 10.3 against 7.6).
bool short_k(const LpArgs& x, bool vec) {
  return x.k < (vec ? 64 : 8) && tile_count(x.m, x.n, 32, 64) > 1024;
}

template <typename T, typename OutT>
int launch_short_k(const LpArgs& x, bool vec) {
  const int64_t tiles = tile_count(x.m, x.n, 128, 128), rounds = (tiles + 255) / 256;
  if (rounds >= 2 && 10 * tiles >= 8 * 256 * rounds)
    return launch_staged<T, OutT, 128, 128>(x, vec);
  return launch_staged<T, OutT, 64, 64>(x, vec);
}

// The WHOLE form.
template <typename T, typename OutT, int BM, int BN>
int launch_whole(const LpArgs& x) {
  const int64_t tiles = tile_count(x.m, x.n, BM, BN);
  if (int rc = check_grid(tiles, kMfmaThreads)) return rc;
  gemm_lp_kernel<T, OutT, BM, BN, false, true>
      <<<static_cast<unsigned>(tiles), kMfmaThreads, 0, x.s>>>(
          x.a, x.b, static_cast<OutT*>(x.c), x.m, x.n, x.k, x.alpha, x.beta,
          steps_along(x.m, BM), steps_along(x.n, BN));
  MCKE_LAUNCH_CHECK("gemm_lp_kernel");
  return ok();
}

template <typename T, typename OutT, int BM, int BN>
int launch_dma32(const LpArgs& x) {
  constexpr int kStages = 4;
  const int64_t tiles = tile_count(x.m, x.n, BM, BN);
  if (int rc = check_grid(tiles, kMfmaThreads)) return rc;
  gemm_lp_dma_kernel<T, OutT, BM, BN, kStages>
      <<<static_cast<unsigned>(tiles), kMfmaThreads, 0, x.s>>>(
          x.a, x.b, static_cast<OutT*>(x.c), x.m, x.n, x.k, x.alpha, x.beta, x.m / BM, x.n / BN);
  MCKE_LAUNCH_CHECK("gemm_lp_dma_kernel");
  return ok();
}

// The EDGE form at BM x BN, where the shape and the addresses allow it.
template <int BM, int BN> bool edge_fits(const LpArgs& x) {
  return x.n >= BN && x.k >= 64 && x.n % 2 == 0 && x.k % 2 == 0 && aligned(x.a, 4) &&
         aligned(x.b, 4) && aligned(x.c, 4) && dma_offsets32<BM, BN>(x.n, x.k);
}

// The register-staged kernel's WHOLE form at BM x BN, where the shape and the addresses
// allow it.
template <int BM, int BN, typename OutT> bool whole_fits(const LpArgs& x) {
  return x.n >= BN && x.k >= 64 && aligned(x.a, 2) && aligned(x.b, 2) &&
         aligned(x.c, sizeof(OutT));
}

template <typename T, typename OutT, int BM, int BN>
struct LpTile {
  // Whole tiles run the requested tile's direct-to-LDS kernel (tiles of 128 and more).
  // Other shapes run its EDGE form, at 128 x 128 from 208 such tiles on, or from 80 on where
  // K is long enough to pay for a tile alone on its CU, and at 256 x 256 where they nearly
  // fill the CUs (fp16 to fp32: 2757 x 432 x 6080, 88 tiles of 128, 49.8 us against 56.9 for
  // split K; 1628 x 800 x 1110, 91 tiles, 15.9 against 15.2; 300 x 520 x 1032, 15 tiles, 14.4
  // against 7.6; 4524 x 344 x 96, 108 tiles, 7.5 against 5.8, to fp16 5.9 against 5.5;
  // 4095 x 4094 x 4090, 256 tiles of 256, 126 us against 206 at 128).  Odd extents run the
  // register-staged kernel's WHOLE form where its 128 x 128 tiles fill most of the CUs (a tile
  // alone on its CU takes 1.3 us per 64 of K, so fewer lose to split K: 1531 x 1021 x 2053, 96
  // tiles, 44.4 us against 29.9; 1700 x 1701 x 1024, 196 tiles, 24.0 against 20.8;
  // 4032 x 843 x 2744, 224 tiles, 54.5 against 63.9; 1901 x 2001 x 511, 240 tiles, 20.4 against
  // 22.1; 3001 x 2501 x 901, 480 tiles, 33.1 against 50.0), at 256 x 256 from 192 such tiles on
  // (4095^3 199 us against 229 at 128 and 406 for split K; 3500 x 3501 x 2001, 196 tiles, 99
  // against 105).  What is left takes the split-K kernel, as 64 x 64 launches do, but for
  // short K over many tiles (short_k).  The tile counts here and below are for 256 CUs.
  static int launch(const LpArgs& x, bool vec) {
    if constexpr (BN >= 128) {
      if (vec && x.m % BM == 0 && x.n % BN == 0 && x.k % 64 == 0 && x.k > 0 &&
          dma_offsets32<BM, BN>(x.n, x.k))
        return launch_dma<T, OutT, BM, BN, false>(x);
      if constexpr (BM == 128)
        if (vec && x.m % BM == 0 && x.n % BN == 0 && x.k % 64 == 32 &&
            tile_count(x.m, x.n, BM, BN) >= 80 && dma_offsets32<BM, BN>(x.n, x.k))
          return launch_dma32<T, OutT, BM, BN>(x);
      if constexpr (BM == 256)
        if (edge_fits<256, 256>(x) && tile_count(x.m, x.n, 256, 256) >= 192)
          return launch_dma<T, OutT, 256, 256, true>(x);
      const int64_t tiles = tile_count(x.m, x.n, 128, 128);
      if (edge_fits<128, 128>(x) &&
          (tiles >= 208 || (tiles >= 80 && x.k >= (sizeof(OutT) == 4 ? 256 : 100))))
        return launch_dma<T, OutT, 128, 128, true>(x);
      if constexpr (BM == 256)
        if (whole_fits<256, 256, OutT>(x) && tile_count(x.m, x.n, 256, 256) >= 192)
          return launch_whole<T, OutT, 256, 256>(x);
      if (whole_fits<128, 128, OutT>(x) && tiles >= 208)
        return launch_whole<T, OutT, 128, 128>(x);
    }
    // 16-bit values at 2-byte addresses, per-lane offsets below 4 GiB, and a grid that holds
    // 32 x 32 tiles of 512 lanes.
    if (x.n >= 32 && x.k > 0 && tile_count(x.m, x.n, 32, 32) <= int64_t{UINT32_MAX} / 512 &&
        aligned(x.a, 2) && aligned(x.b, 2) && aligned(x.c, sizeof(OutT)) &&
        static_cast<int64_t>(64) * x.k * 2 < (int64_t{1} << 32) &&
        static_cast<int64_t>(64) * x.n * 2 < (int64_t{1} << 32))
      return short_k(x, vec) ? launch_short_k<T, OutT>(x, vec) : launch_split<T, OutT>(x);
    return launch_staged<T, OutT, BM, BN>(x, vec);
  }
  // The instantiation whole-tile shapes run, for attribute queries.
  static LpKernel kernel() {
    if constexpr (BN >= 128)
      return reinterpret_cast<LpKernel>(&gemm_lp_dma16_kernel<T, OutT, BM, BN, false>);
    else
      return reinterpret_cast<LpKernel>(&gemm_lp_split_kernel<T, OutT, 4, 4, 4>);
  }
};

// Instantiated tiles: (bm, bn) with bk = 64 and 256 lanes, so (tm, tn) = (bm/16, bn/16).
constexpr int kLpTiles[][2] = {{256, 256}, {128, 128}, {64, 64}};

int lp_tile_index(const mcke_gemm_tile* t) {
  if (!t) return -1;
  for (int i = 0; i < 3; ++i) {
    const int bm = kLpTiles[i][0], bn = kLpTiles[i][1];
    if (t->bm == bm && t->bn == bn && t->bk == kLpBK && t->tm == bm / 16 && t->tn == bn / 16)
      return i;
  }
  return -1;
}

template <typename T, typename OutT>
struct LpTable {
  static int launch(int ti, const LpArgs& x, bool vec) {
    switch (ti) {
      case 0: return LpTile<T, OutT, 256, 256>::launch(x, vec);
      case 1: return LpTile<T, OutT, 128, 128>::launch(x, vec);
      default: return LpTile<T, OutT, 64, 64>::launch(x, vec);
    }
  }
  static LpKernel kernel(int ti) {
    switch (ti) {
      case 0: return LpTile<T, OutT, 256, 256>::kernel();
      case 1: return LpTile<T, OutT, 128, 128>::kernel();
      default: return LpTile<T, OutT, 64, 64>::kernel();
    }
  }
};

// (ab_dtype, c_dtype) -> 0..3, or -1 when the pair is not supported.
int lp_combo(int ab, int cd) {
  if (ab == MCKE_DTYPE_BF16) return cd == MCKE_DTYPE_F32 ? 0 : cd == MCKE_DTYPE_BF16 ? 1 : -1;
  if (ab == MCKE_DTYPE_F16) return cd == MCKE_DTYPE_F32 ? 2 : cd == MCKE_DTYPE_F16 ? 3 : -1;
  return -1;
}

int check_combo(const char* who, int ab, int cd, int* combo) {
  if (ab != MCKE_DTYPE_BF16 && ab != MCKE_DTYPE_F16)
    return invalid(std::string(who) + ": ab_dtype must be MCKE_DTYPE_BF16 or MCKE_DTYPE_F16, got " +
                   std::to_string(ab));
  *combo = lp_combo(ab, cd);
  if (*combo < 0)
    return invalid(std::string(who) + ": c_dtype must be MCKE_DTYPE_F32 or ab_dtype, got " +
                   std::to_string(cd));
  return ok();
}

int check_tile(const char* who, const mcke_gemm_tile* tile, int* ti) {
  *ti = lp_tile_index(tile);
  if (*ti < 0)
    return invalid(std::string(who) +
                   ": instantiated for tiles (bm,bn,bk,tm,tn) = (256,256,64,16,16), "
                   "(128,128,64,8,8) and (64,64,64,4,4); no fallback is applied");
  return ok();
}

}  // namespace
}  // namespace mcke_amd

using namespace mcke_amd;

extern "C" {

int mcke_launch_gemm_lp(const void* a, const void* b, void* c, int ab_dtype, int c_dtype,
                        int64_t m, int64_t n, int64_t k, float alpha, float beta,
                        const mcke_gemm_tile* tile, void* stream) {
  int combo = -1, ti = -1;
  if (int rc = check_combo("launch_gemm_lp", ab_dtype, c_dtype, &combo)) return rc;
  if (int rc = check_tile("launch_gemm_lp", tile, &ti)) return rc;
  if (m == 0 || n == 0) return ok();
  if (m < 0 || n < 0 || k < 0) return invalid("launch_gemm_lp: negative extent");
  if (!a || !b || !c) return invalid("launch_gemm_lp: null pointer");
  if (a == c || b == c)
    return invalid("launch_gemm_lp: output aliases an input, which violates the "
                   "__restrict__ contract");
  if (m > 2147483647LL || n > 2147483647LL || k > 2147483647LL)
    return invalid("launch_gemm_lp: extent exceeds INT32_MAX");
  // 16-byte loads of eight elements need k % 8, n % 8 and 16-byte aligned bases;
  // the C vector stores need C 16-byte aligned as well.
  const bool vec = (k % 8 == 0) && (n % 8 == 0) && aligned(a, 16) && aligned(b, 16) &&
                   aligned(c, 16);
  const LpArgs x{static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b), c,
                 static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), alpha, beta,
                 static_cast<hipStream_t>(stream)};
  switch (combo) {
    case 0: return LpTable<__bf16, float>::launch(ti, x, vec);
    case 1: return LpTable<__bf16, __bf16>::launch(ti, x, vec);
    case 2: return LpTable<_Float16, float>::launch(ti, x, vec);
    default: return LpTable<_Float16, _Float16>::launch(ti, x, vec);
  }
}

int mcke_gemm_lp_kernel_attrs(int ab_dtype, int c_dtype, const mcke_gemm_tile* tile,
                              mcke_kernel_attrs* out) {
  if (!out) return invalid("gemm_lp_kernel_attrs: null out");
  int combo = -1, ti = -1;
  if (int rc = check_combo("gemm_lp_kernel_attrs", ab_dtype, c_dtype, &combo)) return rc;
  if (int rc = check_tile("gemm_lp_kernel_attrs", tile, &ti)) return rc;
  LpKernel kern = nullptr;
  switch (combo) {
    case 0: kern = LpTable<__bf16, float>::kernel(ti); break;
    case 1: kern = LpTable<__bf16, __bf16>::kernel(ti); break;
    case 2: kern = LpTable<_Float16, float>::kernel(ti); break;
    default: kern = LpTable<_Float16, _Float16>::kernel(ti); break;
  }
  hipFuncAttributes fa{};
  MCKE_HIP_TRY(hipFuncGetAttributes(&fa, kern));
  out->regs_per_thread = fa.numRegs;
  out->agprs_per_thread = 0;
  out->static_smem_bytes = fa.sharedSizeBytes;
  out->local_bytes = fa.localSizeBytes;
  out->threads_per_block = kMfmaThreads;
  int blocks = 0;
  MCKE_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kern, kMfmaThreads, 0));
  out->max_blocks_per_sm_api = blocks;
  return ok();
}

int mcke_gemm_lp_default_tile(int64_t m, int64_t n, int64_t k, mcke_gemm_tile* out) {
  if (!out) return invalid("gemm_lp_default_tile: null out");
  (void)k;
  // The largest tile that still fills most of a 256-CU part.  Measured on MI355X: 256 x 256
  // wins at 4096^3 (256 tiles) and at 3072 x 4096 x 1024 (192 tiles, bf16: 32.1 us against
  // 33.6), 128 x 128 at 2048^3 (256 tiles: 23.2 us against 37.2 for 64 x 64) and down to
  // 80 tiles (a launch of fewer than 208 that are not whole still splits K where K is short or
  // odd), 64 x 64 at 1024^3 (64 tiles of 128: 12.4 us against 8.8).
  auto tiles = [&](int64_t t) { return ((m + t - 1) / t) * ((n + t - 1) / t); };
  if (tiles(256) >= 192) *out = mcke_gemm_tile{256, 256, kLpBK, 16, 16};
  else if (tiles(128) >= 80) *out = mcke_gemm_tile{128, 128, kLpBK, 8, 8};
  else *out = mcke_gemm_tile{64, 64, kLpBK, 4, 4};
  return ok();
}

}  // extern "C"
