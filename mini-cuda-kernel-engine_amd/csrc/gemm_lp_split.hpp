// gemm_lp_split.hpp -- 16-bit-input GEMM whose waves split K: C = alpha A B + beta C,
// row-major, bf16 or fp16 in, fp32 accumulation, fp32 or 16-bit C; any M, any N >= the
// tile's width, any K, any element alignment.
//
// For tiles up to 64 x 64 and for shapes that fill too few CUs with larger ones.  With a
// tile this small a 2 x 2 wave grid reads each operand from LDS twice (256 bytes per
// cycle at 64 x 64 for 16x16x32 MFMAs, twice what LDS delivers) and meets at a barrier
// for a few MFMAs' worth of work.  Here
//   * every wave computes the whole 16 MT x 16 NW tile over its own K chunks (32 deep, dealt
//     to the WV waves in turn), so a fragment is read from LDS once, and the loop has no
//     barrier: a wave loads a chunk into registers, writes it to an LDS slot of its own while
//     the next chunk's loads are in flight, and reads the fragments back;
//   * loads are 16 bytes per lane at 2-byte alignment, so odd widths and unaligned
//     operands take the same path (the register-staged kernel loads them 2 bytes at a
//     time);
//   * B is transposed by the LDS (ds_read_b64_tr_b16) on the way back;
//   * the waves' sums are folded through LDS in a fixed order at the end.
//
// Measured on MI355X, fp16 to fp32, four sets of operands in turn (us; the
// register-staged kernel, 64 x 64 tile, then this one in the configuration that the
// launcher picks):
//   16 x 32, 8 waves:  16 x 4096 x 4096  46.5  12.1    9 x 5184 x 1523     58.9   5.7
//   32 x 32, 8 waves:  32 x 4096 x 4096  47.1  13.8
//   32 x 64, 4 waves:  64 x 4096 x 4096  47.5  15.7    1024^3              15.4   8.6
//                      36 x 7379 x 8064   411  45.9    317 x 304 x 960     12.5   5.5
//                      1628 x 800 x 1109 77.4  15.6    1531 x 1021 x 2053   123  29.4
//   64 x 64, 4 waves:  1700 x 1501 x 1024  85.8  20.4
// Direct-to-LDS loads in the same scheme are within 6% either way (16 x 4096 x 4096 12.4
// against 11.8 in one sweep, 1024^3 7.9 against 8.4) and need 4-byte alignment.
//
// LDS slot of a wave, per chunk: 1 KB per 16 rows of A, rows of 64 bytes with 16-byte quad q
// of row r at q ^ aswz(r); NW KB of B: k = 8 g + 4 t + j sits at position
// s = 16 t + 4 g + j (a transposed read takes one t), 32-byte column block b of a position
// at b ^ bswz(s).  Both put what a half-wave reads on distinct banks.
#pragma once

#include "gemm_lp.hpp"

namespace mcke_amd {

typedef short s16x4 __attribute__((ext_vector_type(4)));

template <int MT, int NW, int WV>
struct LpSplitShape {
  static constexpr int TM = 16 * MT, TN = 16 * NW;
  static constexpr int KC = 32;                           // K per chunk
  static constexpr int NA = MT, NB = NW;                  // 1 KB loads per chunk
  static constexpr int L = NA + NB;
  static constexpr int kSlot = L * 1024;
  static constexpr int kThreads = WV * 64;
  static constexpr int kSlots = WV * kSlot;
  static constexpr int kOut = TM * TN;                    // values of one wave's sums
  // How many waves' sums fit beside each other: a power of two, all of them if that
  // takes no more LDS than the slots.
  static constexpr int kFold = kOut * 4 * WV <= kSlots ? WV : WV / 2;
  static constexpr int kLds = kSlots > kFold * kOut * 4 ? kSlots : kFold * kOut * 4;
  static_assert(kLds <= 64 * 1024, "two workgroups or more per CU");
  static constexpr int kARow = 64, kBRow = 32 * NW;
  static_assert(NW == 2 || NW == 4, "column blocks are swizzled in twos or fours");
  static __host__ __device__ constexpr int aswz(int r) { return (r >> 2) & 3; }
  static __host__ __device__ constexpr int bswz(int s) {
    return NW == 2 ? (s >> 2) & 1 : (s >> 1) & 3;
  }
};

template <typename T, typename OutT, int MT, int NW, int WV>
__global__ __launch_bounds__(WV * 64) void gemm_lp_split_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, OutT* __restrict__ C, int M,
    int N, int K, float alpha, float beta, int tiles_m, int tiles_n) {
  using S = LpSplitShape<MT, NW, WV>;
  constexpr int L = S::L;
  __shared__ __attribute__((aligned(1024))) char smem[S::kLds];

  int tm, tn;
  mfma_tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * S::TM, n_first = tn * S::TN;
  const int n0 = n_first > N - S::TN ? N - S::TN : n_first;

  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int g = lane / 16, c = lane % 16;

  // Source byte offsets of this lane's 16 bytes in each 1 KB load of a chunk (the launcher
  // keeps them in 32 bits).  Rows past M repeat row M - 1 and are not stored; the last tile
  // column starts at N - TN and stores only the columns of its own.
  // a_k and b_k: the first k of the lane's eight in A, and its k in B.
  uint32_t a_src[S::NA], b_src[S::NB];
  int b_k[S::NB];
  const int a_row = lane / 4, a_quad = (lane % 4) ^ S::aswz(a_row), a_k = 8 * a_quad;
#pragma unroll
  for (int i = 0; i < S::NA; ++i) {
    const int row_t = 16 * i + a_row;
    const int row = row_t > M - 1 - m0 ? M - 1 - m0 : row_t;
    a_src[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(K) * 2u + 16u * a_quad;
  }
#pragma unroll
  for (int u = 0; u < S::NB; ++u) {
    const int at = u * 1024 + 16 * lane;
    const int s = at / S::kBRow;
    const int b = ((at % S::kBRow) / 32) ^ S::bswz(s);
    b_k[u] = 8 * ((s / 4) % 4) + 4 * (s / 16) + s % 4;
    b_src[u] = (static_cast<uint32_t>(b_k[u]) * static_cast<uint32_t>(N) + 16u * b) * 2u +
               static_cast<uint32_t>(at % 32);
  }
  const char* a_base = reinterpret_cast<const char*>(A + static_cast<int64_t>(m0) * K);
  const char* b_base = reinterpret_cast<const char*>(B + n0);
  char* slot = smem + wave * S::kSlot;

  // Fragment addresses within a slot.
  const uint32_t a_off = c * S::kARow + 16 * (g ^ S::aswz(c));
  uint32_t b_off[NW];
#pragma unroll
  for (int b = 0; b < NW; ++b) {
    const int s = g * 4 + c / 4;                        // read t adds 16 positions
    b_off[b] = S::NA * 1024 + s * S::kBRow + 32 * (b ^ S::bswz(s)) + 8 * (c % 4);
  }

  f32x4 acc[MT][NW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int b = 0; b < NW; ++b) acc[i][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int chunks = K / S::KC;
  const int n_it = chunks > wave ? (chunks - wave + WV - 1) / WV : 0;
  auto compute = [&]() {
    u32x4 av[MT];
    u32x2 bv[NW][2];
#pragma unroll
    for (int m = 0; m < MT; ++m) av[m] = *reinterpret_cast<const u32x4*>(slot + m * 1024 + a_off);
#pragma unroll
    for (int b = 0; b < NW; ++b)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        bv[b][t] = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                       (__attribute__((address_space(3))) s16x4*)(
                           slot + t * (16 * S::kBRow) + b_off[b])));
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int bb = 0; bb < NW; ++bb) {
        const int b = mfma_snake_col(m, bb, NW);
        acc[m][b] = LpMfma16<T>::run(
            av[m], u32x4{bv[b][0][0], bv[b][0][1], bv[b][1][0], bv[b][1][1]}, acc[m][b]);
      }
  };

  auto load = [&](int it, u32x4 (&v)[L]) {
    const int64_t k0 = static_cast<int64_t>(S::KC) * (wave + WV * it);
    const char* ap = a_base + k0 * 2;
    const char* bp = b_base + k0 * N * 2;
#pragma unroll
    for (int i = 0; i < S::NA; ++i) v[i] = *reinterpret_cast<const u32x4_a2*>(ap + a_src[i]);
#pragma unroll
    for (int u = 0; u < S::NB; ++u)
      v[S::NA + u] = *reinterpret_cast<const u32x4_a2*>(bp + b_src[u]);
  };
  auto to_slot = [&](const u32x4 (&v)[L]) {
#pragma unroll
    for (int i = 0; i < L; ++i) *reinterpret_cast<u32x4*>(slot + i * 1024 + 16 * lane) = v[i];
  };
  // Lanes read what other lanes of the wave wrote.
  auto written = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  // K's remainder is a chunk of the wave whose turn it is, its first one, zero past the end
  // in both operands; its loads and those of the next chunk are in flight together.  An eight
  // of A that the end cuts is the row's last eight, shifted into place (rows of less than
  // eight: element by element).  Loaded element by element as a whole, after the loop, the
  // remainder took up to 1.8 us, much of a short product's time: fp16 to fp16, 33 x 2200 x 16
  // 5.7 -> 4.1 us, 2460 x 1608 x 40 14.9 -> 10.7.
  u32x4 v[L];
  const int rem = K % S::KC;
  if (rem != 0 && wave == chunks % WV) {
    const int past = 8 - rem % 8;        // of a cut eight, what lies past the end
    const int64_t k0 = static_cast<int64_t>(S::KC) * chunks;
    const char* ap = a_base + k0 * 2;
    const char* bp = b_base + k0 * N * 2;
    u32x4 w[L];
#pragma unroll
    for (int i = 0; i < S::NA; ++i) {
      w[i] = u32x4{0u, 0u, 0u, 0u};
      if (a_k + 8 <= rem) {
        w[i] = *reinterpret_cast<const u32x4_a2*>(ap + a_src[i]);
      } else if (a_k < rem) {
        if (K >= 8) {
          const u32x4 last8 = *reinterpret_cast<const u32x4_a2*>(ap + a_src[i] - 2 * past);
          w[i] =
              __builtin_bit_cast(u32x4, __builtin_bit_cast(unsigned __int128, last8) >> (16 * past));
        } else {
          w[i] = lp_load8<false>(reinterpret_cast<const uint16_t*>(ap + a_src[i]), a_k, rem, true);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < S::NB; ++u) {
      w[S::NA + u] = u32x4{0u, 0u, 0u, 0u};
      if (b_k[u] < rem) w[S::NA + u] = *reinterpret_cast<const u32x4_a2*>(bp + b_src[u]);
    }
    if (n_it > 0) load(0, v);
    to_slot(w);
    written();
    compute();
  } else if (n_it > 0) {
    load(0, v);
  }
  for (int it = 0; it < n_it; ++it) {
    // The slot's last reads have been waited for by the MFMAs that used them.
    to_slot(v);
    load(it + 1 < n_it ? it + 1 : it, v);
    written();
    compute();
  }

  // The waves' sums.  While there are more than fit, the upper half hands its own to the
  // lower half; then kFold of them lie side by side and every lane adds them up for the
  // outputs it stores.  Lane (g, c), register r of block (m, b): row 16 m + 4 g + r,
  // column 16 b + c.
  float* sums = reinterpret_cast<float*>(smem);
  auto at = [&](int w, int m, int b, int r) {
    return w * S::kOut + ((m * NW + b) * 4 + r) * 64 + lane;
  };
  auto put = [&](int w) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int b = 0; b < NW; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[at(w, m, b, r)] = acc[m][b][r];
  };
  __syncthreads();
  if constexpr (S::kFold < WV) {
    static_assert(2 * S::kFold == WV, "one hand-over");
    if (wave >= S::kFold) put(wave - S::kFold);
    __syncthreads();
    if (wave < S::kFold) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int b = 0; b < NW; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][b][r] += sums[at(wave, m, b, r)];
    }
    // Each wave overwrites only the sums that it has just read.
  }
  if (wave < S::kFold) put(wave);
  __syncthreads();
  using O = LpOut<OutT>;
  struct Pack { OutT v[4]; };   // four adjacent columns at any address
  for (int q = threadIdx.x; q < S::kOut / 4; q += S::kThreads) {
    const int rt = q / (S::TN / 4), cq = q % (S::TN / 4);
    const int row = m0 + rt, col = n0 + 4 * cq;
    if (row >= M || col + 3 < n_first) continue;
    const int o = (((rt / 16) * NW + cq / 4) * 4 + rt % 4) * 64 + 16 * ((rt / 4) % 4) + 4 * (cq % 4);
    f32x4 s = *reinterpret_cast<const f32x4*>(sums + o);
#pragma unroll
    for (int w = 1; w < S::kFold; ++w)
      s += *reinterpret_cast<const f32x4*>(sums + w * S::kOut + o);
    OutT* p = C + static_cast<int64_t>(row) * N + col;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] *= alpha;
      if (beta != 0.0f && col + j >= n_first) s[j] += beta * O::to_f32(p[j]);
    }
    if (col >= n_first) {
      Pack out;
#pragma unroll
      for (int j = 0; j < 4; ++j) out.v[j] = O::from_f32(s[j]);
      __builtin_memcpy(p, &out, sizeof(out));
    } else {
#pragma unroll
      for (int j = 1; j < 4; ++j)
        if (col + j >= n_first) p[j] = O::from_f32(s[j]);
    }
  }
}

}  // namespace mcke_amd
