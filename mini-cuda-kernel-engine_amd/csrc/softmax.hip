// softmax.hip -- numerically stable row softmax.
//
// Replaces kernels/softmax.cu (launcher softmax.cu:177-199, kernels :112-173,
// online combine :77-107) on top of the (m, d) algebra of
// include/mcke/kernels/softmax_online.hpp:73-112.
//
// kOnlineOnePass is the fast path and is HBM-bound at the compulsory traffic of
// one read and one write per element (2 * rows * cols * 4 bytes):
//   * rows that fit in registers (up to 65539 columns, any width and 4-byte
//     alignment) are held in VGPRs: a group of TPR lanes owns a row, each lane
//     loads VPT float4s, the group reduces the max and then sum(exp(x-m))
//     by wave64 butterflies (plus one LDS stage when a row spans several waves),
//     and the row is written from the same registers -- 1R + 1W;
//   * longer rows fall back to the reference's online form: one traversal
//     carrying (m, d) per lane, a workgroup combine, and a write pass -- 2R + 1W.
// kThreePass is the baseline: max pass, sum pass, write pass (3R + 1W).
//
// exp(t) for t = x - m <= 0 is evaluated as 2^(t * log2 e) with the hardware
// exponential; the product's rounding perturbs the result by at most |t| * 2^-24
// relative, which is below 1e-9 in absolute terms wherever exp(t) is not already
// negligible.  The row's 1/d is one correctly rounded division per row.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <string>

#include "common.hpp"
#include "device_math.hpp"

namespace mcke_amd {
namespace {

constexpr int kThreads = 256;
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float exp_le0(float t) {
  return __builtin_amdgcn_exp2f(t * kLog2e);
}

// ---------------------------------------------------------------------------
// Register-resident rows.  NT-lane workgroups, TPR lanes per row (8 .. 1024), VPT
// float4 per lane.  A row wider than a wave spans TPR / 64 consecutive waves,
// combined through one LDS stage over that row's own waves.
// ---------------------------------------------------------------------------
// A row over TPR / 64 waves: each wave's result in LDS, then every wave folds the row's
// results by a butterfly of its own (waves are a power of two).  The butterfly adds them
// as a tree: added one after the other, the small terms beside a row's dominant one were
// rounded away up to 15 times instead of 4.
template <int TPR> __device__ __forceinline__ float group_max(float v, float* lds) {
  if constexpr (TPR <= kWave) {
    return wave_max<TPR>(v);
  } else {
    constexpr int W = TPR / kWave;
    v = wave_max<kWave>(v);
    const int first = (threadIdx.x / TPR) * W;   // the row's first wave
    if ((threadIdx.x % kWave) == 0) lds[threadIdx.x / kWave] = v;
    __syncthreads();
    const float r = wave_max<W>(lds[first + threadIdx.x % W]);
    __syncthreads();   // lds is reused by group_sum
    return r;
  }
}

template <int TPR> __device__ __forceinline__ float group_sum(float v, float* lds) {
  if constexpr (TPR <= kWave) {
    return wave_sum<TPR>(v);
  } else {
    constexpr int W = TPR / kWave;
    v = wave_sum<kWave>(v);
    const int first = (threadIdx.x / TPR) * W;
    if ((threadIdx.x % kWave) == 0) lds[threadIdx.x / kWave] = v;
    __syncthreads();
    return wave_sum<W>(lds[first + threadIdx.x % W]);
  }
}

// ALIGNED: every row of x and y starts on 16 bytes and cols % 4 == 0.  Otherwise a row
// is split at y's 16-byte boundaries: `head` (0 .. 3) elements before the first one,
// whole vectors, `tail` (0 .. 3) elements after the last one; the up to six edge
// elements are one float in each of the row's first lanes (TPR >= 8).  Stores of whole
// vectors are then aligned for any width; loads of x take 4-byte alignment.
template <int TPR, int VPT, int NT, bool ALIGNED>
__global__ __launch_bounds__(NT) void softmax_regs_kernel(const float* __restrict__ x,
                                                          float* __restrict__ y, int64_t rows,
                                                          int64_t cols) {
  static_assert(NT % TPR == 0, "TPR must divide the workgroup");
  static_assert(TPR >= 8, "the edge elements take one lane each");
  constexpr int kRowsPerBlock = NT / TPR;
  // Neighbouring short rows share cache lines when they are not line-aligned, so these
  // loads leave the lines in cache: 65536 rows, 129 columns 11.4 vs 13.2 us with
  // streaming loads, 250 columns 20.7 vs 24.1; 4095 columns are slower that way (185 vs
  // 173 at 32768 rows).
  constexpr bool kPlainLoads = !ALIGNED && TPR * VPT <= 64;
  __shared__ float lds[NT / kWave];
  const int t = threadIdx.x % TPR;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + threadIdx.x / TPR;
  // Rows past the end still take part in the barriers of a multi-wave group,
  // so they only skip their loads and stores.  (With TPR <= 64 a whole group is
  // one wave and there are no barriers.)
  const bool live = r < rows;
  const float* __restrict__ xrow = x + (live ? r : 0) * cols;
  float* __restrict__ yrow = y + (live ? r : 0) * cols;

  // At most VPT * TPR vectors: within 32 bits.
  const int n = static_cast<int>(cols);
  int head = 0;
  if constexpr (!ALIGNED) {
    head = static_cast<int>((0 - (reinterpret_cast<uintptr_t>(yrow) >> 2)) & 3);
    head = head < n ? head : n;
  }
  const int cols_v = (n - head) >> 2;
  const float* __restrict__ xr = xrow + head;
  f32x4* __restrict__ yr = reinterpret_cast<f32x4*>(yrow + head);

  f32x4 v[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int j = i * TPR + t;
    if (live && j < cols_v) {
      if constexpr (ALIGNED) v[i] = ld_stream(reinterpret_cast<const f32x4*>(xr) + j);
      else v[i] = kPlainLoads ? ld4(xr + 4 * j) : ld_stream4(xr + 4 * j);
    } else {
      v[i] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
  }
  // This lane's edge element: head element t, or tail element t - head.
  float e = -INFINITY;
  int ei = t;
  bool has_e = false;
  if constexpr (!ALIGNED) {
    const int edges = n - 4 * cols_v;
    if (t >= head) ei = t + 4 * cols_v;
    has_e = live && t < edges;
    if (has_e) e = ld_stream(xrow + ei);
  }
  float m = e;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    m = fmaxf(m, fmaxf(fmaxf(v[i][0], v[i][1]), fmaxf(v[i][2], v[i][3])));
  m = group_max<TPR>(m, lds);

  float d = 0.0f;
  if constexpr (!ALIGNED) {
    if (has_e) {
      e = exp_le0(e - m);
      d = e;
    }
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int j = i * TPR + t;
    if (j < cols_v) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[i][c] = exp_le0(v[i][c] - m);
        d += v[i][c];
      }
    }
  }
  d = group_sum<TPR>(d, lds);
  const float inv = 1.0f / d;
  if (!live) return;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int j = i * TPR + t;
    if (j < cols_v) st_stream(yr + j, v[i] * inv);
  }
  if constexpr (!ALIGNED) {
    if (has_e) st_stream(yrow + ei, e * inv);
  }
}

// ---------------------------------------------------------------------------
// Online (m, d) fallback and the three-pass baseline: one workgroup per row.
// ---------------------------------------------------------------------------
struct OnlineState {
  float m, d;
};

__device__ __forceinline__ OnlineState online_identity() { return {-FLT_MAX, 0.0f}; }

__device__ __forceinline__ OnlineState online_update(OnlineState s, float x) {
  const float mn = fmaxf(s.m, x);
  return {mn, s.d * exp_le0(s.m - mn) + exp_le0(x - mn)};
}

__device__ __forceinline__ OnlineState online_combine(OnlineState a, OnlineState b) {
  if (b.d == 0.0f) return a;
  if (a.d == 0.0f) return b;
  const float mm = fmaxf(a.m, b.m);
  return {mm, a.d * exp_le0(a.m - mm) + b.d * exp_le0(b.m - mm)};
}

__device__ __forceinline__ OnlineState block_online(OnlineState s) {
  __shared__ float pm[kThreads / kWave], pd[kThreads / kWave];
#pragma unroll
  for (int k = kWave / 2; k >= 1; k >>= 1) {
    OnlineState o{__shfl_xor(s.m, k, 64), __shfl_xor(s.d, k, 64)};
    s = online_combine(s, o);
  }
  const int w = threadIdx.x / kWave;
  if ((threadIdx.x % kWave) == 0) {
    pm[w] = s.m;
    pd[w] = s.d;
  }
  __syncthreads();
  OnlineState r{pm[0], pd[0]};
#pragma unroll
  for (int i = 1; i < kThreads / kWave; ++i) r = online_combine(r, OnlineState{pm[i], pd[i]});
  return r;
}

__global__ __launch_bounds__(kThreads) void softmax_online_kernel(const float* __restrict__ x,
                                                                  float* __restrict__ y,
                                                                  int64_t cols) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * cols;
  OnlineState s = online_identity();
  for (int64_t c = threadIdx.x; c < cols; c += kThreads) s = online_update(s, x[base + c]);
  s = block_online(s);
  const float inv = 1.0f / s.d;
  for (int64_t c = threadIdx.x; c < cols; c += kThreads)
    y[base + c] = exp_le0(x[base + c] - s.m) * inv;
}

__device__ __forceinline__ float block_max(float v) {
  __shared__ float part[kThreads / kWave];
  v = wave_max(v);
  if ((threadIdx.x % kWave) == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  float r = part[0];
#pragma unroll
  for (int i = 1; i < kThreads / kWave; ++i) r = fmaxf(r, part[i]);
  return r;
}

__device__ __forceinline__ float block_sum(float v) {
  __shared__ float part[kThreads / kWave];
  v = wave_sum(v);
  if ((threadIdx.x % kWave) == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  float r = part[0];
#pragma unroll
  for (int i = 1; i < kThreads / kWave; ++i) r += part[i];
  return r;
}

__global__ __launch_bounds__(kThreads) void softmax_three_pass_kernel(
    const float* __restrict__ x, float* __restrict__ y, int64_t cols) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * cols;
  float m = -INFINITY;
  for (int64_t c = threadIdx.x; c < cols; c += kThreads) m = fmaxf(m, x[base + c]);
  m = block_max(m);
  float d = 0.0f;
  for (int64_t c = threadIdx.x; c < cols; c += kThreads) d += exp_le0(x[base + c] - m);
  d = block_sum(d);
  const float inv = 1.0f / d;
  for (int64_t c = threadIdx.x; c < cols; c += kThreads)
    y[base + c] = exp_le0(x[base + c] - m) * inv;
}

int launch_online_kernel(const float* x, float* y, int64_t rows, int64_t cols, hipStream_t s) {
  softmax_online_kernel<<<static_cast<unsigned>(rows), kThreads, 0, s>>>(x, y, cols);
  MCKE_LAUNCH_CHECK("softmax_online_kernel");
  return ok();
}

// Register-resident configuration for a row of cv whole float4 vectors (plus, for
// rows that are not 16-byte aligned, up to six edge elements).
template <bool ALIGNED, int TPR, int VPT, int NT = kThreads>
int launch_regs(const float* x, float* y, int64_t rows, int64_t cols, hipStream_t s) {
  constexpr int rpb = NT / TPR;
  const int64_t groups = (rows + rpb - 1) / rpb;
  // Wide workgroups of more rows than the grid's 32-bit work size: the online kernel's
  // 256-lane ones go further.
  if (NT > kThreads && groups * NT > int64_t{UINT32_MAX})
    return launch_online_kernel(x, y, rows, cols, s);
  const unsigned g = static_cast<unsigned>(groups);
  softmax_regs_kernel<TPR, VPT, NT, ALIGNED><<<g, NT, 0, s>>>(x, y, rows, cols);
  MCKE_LAUNCH_CHECK("softmax_regs_kernel");
  return ok();
}

template <bool ALIGNED>
int launch_rows(const float* x, float* y, int64_t rows, int64_t cols, hipStream_t s) {
  const int64_t cv = cols / 4;
  if constexpr (ALIGNED) {
    // Short rows: fewer lanes per row and four float4s per lane, so a launch at
    // 32768 rows is one round of resident workgroups with 64 bytes per lane in
    // flight (measured 6.2 us vs 8.2 us for one float4 per lane at 128 columns).
    if (cv <= 32) return launch_regs<true, 8, 4>(x, y, rows, cols, s);
    if (cv <= 64) return launch_regs<true, 16, 4>(x, y, rows, cols, s);
  } else {
    // Unaligned short rows read and write in pieces of their own, so a wave that spans
    // fewer rows at a time does better.  65536 rows: 129 columns 32 x 2 13.2 us, 16 x 4
    // 15.0, 8 x 4 18.9; 131072 x 50: 16 x 1 10.7, 8 x 2 14.6, 32 x 1 16.3; 262144 x 33:
    // 8 x 2 15.4, 16 x 1 16.6.
    if (cv <= 8) return launch_regs<false, 8, 2>(x, y, rows, cols, s);
    if (cv <= 16) return launch_regs<false, 16, 1>(x, y, rows, cols, s);
    if (cv <= 64) return launch_regs<false, 32, 2>(x, y, rows, cols, s);
  }
  // Longer rows: two float4s per lane over more lanes.  At 32768 x 1024, 128
  // lanes x 2 took 42.9 us in 256-lane workgroups and 42.45 in 512-lane ones of
  // four rows (64 x 4: 43.4, 32 x 8: 44.5, 256 x 1: 45.1; a one-wave float4 copy
  // of the same bytes 41.1); at 32768 x 4096, 512-lane workgroups of one
  // row x 2 took 163.2 us (256 x 4: 172.9, 128 x 8: 178.0, 64 x 16: 181.4; the
  // copy 165.5); at 16384 x 8192, 1024-lane workgroups of one row x 2 took
  // 171.0 us (256 x 8: 176.5, 512 x 4: 187.2).  Unaligned rows rank the same: 1023
  // columns 45.2-45.9 us, 4095 columns 172.8-173.9 us at 32768 rows.
  if (cv <= 128) return launch_regs<ALIGNED, 64, 2>(x, y, rows, cols, s);
  if (cv <= 256) return launch_regs<ALIGNED, 128, 2, 512>(x, y, rows, cols, s);
  if (cv <= 512) return launch_regs<ALIGNED, 64, 8>(x, y, rows, cols, s);
  if (cv <= 1024) return launch_regs<ALIGNED, 512, 2, 512>(x, y, rows, cols, s);
  if (cv <= 2048) return launch_regs<ALIGNED, 1024, 2, 1024>(x, y, rows, cols, s);
  // Rows past 8192 columns: one 1024-lane workgroup with 4, 8 or 16 float4s per lane,
  // as far as its registers hold a row.  The online form, which reads x twice, took
  // 397 us at 4096 x 32001 and 220 us at 8192 x 9999; this takes 188-190 us and 107 us
  // (8 per lane and 4 per lane; 512 lanes x 16: 192 and 109), and at 462 x 54889, 16
  // per lane, 43 us for 172.
  if (cv <= 4096) return launch_regs<ALIGNED, 1024, 4, 1024>(x, y, rows, cols, s);
  if (cv <= 8192) return launch_regs<ALIGNED, 1024, 8, 1024>(x, y, rows, cols, s);
  return launch_regs<ALIGNED, 1024, 16, 1024>(x, y, rows, cols, s);
}

// The longest row the register path holds, in float4 vectors.
constexpr int64_t kMaxRegVectors = 16384;

int launch_online(const float* x, float* y, int64_t rows, int64_t cols, hipStream_t s) {
  if (cols / 4 <= kMaxRegVectors) {
    const bool vec = (cols % 4 == 0) && aligned(x, 16) && aligned(y, 16);
    return vec ? launch_rows<true>(x, y, rows, cols, s) : launch_rows<false>(x, y, rows, cols, s);
  }
  return launch_online_kernel(x, y, rows, cols, s);
}

}  // namespace
}  // namespace mcke_amd

using namespace mcke_amd;

extern "C" {

int mcke_launch_row_softmax_f32(const float* x, float* y, int64_t rows, int64_t cols,
                                int variant, void* stream) {
  if (rows == 0 || cols == 0) return ok();
  if (rows < 0 || cols < 0) return invalid("launch_row_softmax_f32: negative extent");
  if (!x || !y) return invalid("launch_row_softmax_f32: null pointer");
  if (x == y)
    return invalid("launch_row_softmax_f32: in-place (x == y) violates the __restrict__ contract");
  if (rows > 2147483647LL)
    return invalid("launch_row_softmax_f32: rows exceeds the grid's x limit");
  if (variant != MCKE_SOFTMAX_THREE_PASS && variant != MCKE_SOFTMAX_ONLINE_ONE_PASS)
    return invalid("launch_row_softmax_f32: unknown SoftmaxVariant");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (variant == MCKE_SOFTMAX_THREE_PASS) {
    softmax_three_pass_kernel<<<static_cast<unsigned>(rows), kThreads, 0, s>>>(x, y, cols);
    MCKE_LAUNCH_CHECK("softmax_three_pass_kernel");
    return ok();
  }
  return launch_online(x, y, rows, cols, s);
}

}  // extern "C"
