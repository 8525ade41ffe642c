// gemm_rows.hpp -- fp32 GEMM for products with few tiles: C = alpha A B + beta C, or the
// fused bias + activation form, row-major.
//
// A product of a few rows is bound by reading B once (4 K N bytes), and a small one by how
// few CUs its tiles reach.  The 32 x 32 tile gives either a workgroup per 32 columns and 32
// rows, four waves each, that meet at a barrier every 32 of K, and spends half or more of
// its MFMA rows on padding if there are 16 rows or less.  Here
//   * a workgroup owns 16 MT rows, W = 16 NW columns and all of K, so that 16 x 4096 is
//     256 workgroups, and its 8 waves take the 32-deep K chunks in turn;
//   * each wave streams its chunks into a ring of its own in LDS by direct-to-LDS loads,
//     with no barrier in the loop (a wave waits for its own loads only);
//   * v_mfma_f32_16x16x4_f32: 16 rows of A per instruction instead of 32;
//   * the waves' sums are added in wave order through LDS at the end.
//
// Measured with four sets of operands in turn (us; the 32 x 32 tile, then this):
//   16 x 4096 x 4096   28.9  15.6 (MT 1, NW 1; a plain read of B takes 10.8)
//   16 x 8192 x 8192   79.5  54.6 (1, 2)      16 x 16384 x 4096  53.6  47.8 (1, 4)
//   32 x 4096 x 4096   29.2  17.1 (1, 2)      64 x 4096 x 4096   29.3  21.7 (2, 2)
//   4 x 259 x 360       4.7   3.3 (1, 1)      96 x 96 x 8000     47.8  17.5 (1, 1)
//   300 x 217 x 4072   27.6  19.3 (1, 2)      512 x 512 x 2048   14.7  11.7 (2, 2)
// Chunks are 32 deep so that A's 128-byte pieces are whole cache lines: every workgroup
// reads all of its rows of A, and with 16-deep chunks (64-byte pieces) the first line took
// 17.2 us.  Rings deeper than two chunks are slower (three: 16.3, four: 16.6): what is in
// flight is enough, and shallow rings keep neighbours, which share lines of B at NW 1,
// together.
//
// Fragments.  One 16x16x4 MFMA takes, per lane l (g = l / 16, c = l % 16), A[c][k_g] and
// B[k_g][c] for the four lane groups' k_g.  MFMA i (0 .. 3) of a chunk's half h uses
// k_g = 16 h + 4 g + i, so a lane's four A values are 16 contiguous bytes of its row.
//
// LDS, per chunk: 2 MT KB of A, rows of 128 bytes with 16-byte quad q of row r at
// q ^ (r % 16) / 2; 2 NW KB of B: row 16 h + 4 g + i sits at position p = 4 i + g of half
// h, 64-byte column block b of a position at b ^ x(p).  The four rows of B that an MFMA
// reads are then neighbours on distinct banks, and so are the quads of A.
//
// Any M (rows past it repeat the last one and are not stored), any N >= W (the last tile
// column starts at N - W and stores only the columns of its own), any K (its last K % 32
// go through registers), 4-byte alignment.
#pragma once

#include "gemm_mfma.hpp"

namespace mcke_amd {

constexpr int kRowsWaves = 8;
constexpr int kRowsThreads = kRowsWaves * 64;
constexpr int kRowsChunk = 32;
constexpr int kRowsDepth = 2;

template <int MT, int NW, bool FUSED>
__global__ __launch_bounds__(kRowsThreads, 1) void gemm_rows_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N,
    int K, float alpha, float beta, int tiles_m, int tiles_n, EpiArgs epi) {
  constexpr int W = 16 * NW;
  constexpr int D = kRowsDepth;
  constexpr int L = 2 * (MT + NW);           // direct-to-LDS instructions per chunk
  static_assert(D >= 2 && (D - 1) * L <= 63, "vmcnt counts at most 63 loads");
  static_assert(NW == 1 || NW == 2 || NW == 4, "column blocks are swizzled in powers of two");
  __shared__ __attribute__((aligned(1024))) char smem[kRowsWaves * D * L * 1024];
  static_assert(MT * NW <= D * L, "the waves' sums must fit in the rings");

  // Neighbouring workgroups share cache lines of B where W is less than a line: each XCD
  // takes a contiguous run of columns.
  int tm, tn;
  mfma_tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * 16 * MT, n_first = tn * W;
  const int n0 = n_first > N - W ? N - W : n_first;
  const int last = M - 1 - m0;               // rows past it repeat it
  A += static_cast<int64_t>(m0) * K;

  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int g = lane / 16, c = lane % 16;

  // Source byte offsets of this lane within a chunk (the launcher keeps them in 32 bits).
  uint32_t a_src[2 * MT], b_src[2 * NW];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int r = 8 * i + lane / 8, row = r < last ? r : last;
    const int quad = (lane % 8) ^ ((r % 16) >> 1);
    a_src[i] = (static_cast<uint32_t>(row) * static_cast<uint32_t>(K) + 4u * quad) * 4u;
  }
  auto swz = [](int p) { return NW == 1 ? 0 : NW == 2 ? (p >> 1) & 1 : p & 3; };
#pragma unroll
  for (int u = 0; u < 2 * NW; ++u) {
    const int at = (u % NW) * 1024 + 16 * lane;
    const int p = at / (64 * NW), b = ((at / 64) % NW) ^ swz(p);
    const int k = 16 * (u / NW) + 4 * (p % 4) + p / 4;
    b_src[u] =
        (static_cast<uint32_t>(k) * static_cast<uint32_t>(N) + 16u * b + (at % 64) / 4u) * 4u;
  }
  const uint32_t lds0 =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
          (const __attribute__((address_space(3))) char*)(smem))) + wave * (D * L * 1024);
  const char* ring = smem + wave * (D * L * 1024);

  const int chunks = K / kRowsChunk;
  const int n_it = chunks > wave ? (chunks - wave + kRowsWaves - 1) / kRowsWaves : 0;
  auto issue = [&](int it, int slot) {
    // Past the end the last chunk is fetched again, which keeps the count of loads in
    // flight uniform.
    const int64_t k0 =
        static_cast<int64_t>(kRowsChunk) * (wave + kRowsWaves * (it < n_it ? it : n_it - 1));
    const uint32_t at = lds0 + slot * (L * 1024);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) lds_dma16<0>(a_src[i], A + k0, at + i * 1024);
#pragma unroll
    for (int u = 0; u < 2 * NW; ++u)
      lds_dma16<0>(b_src[u], B + (k0 * N + n0), at + (2 * MT + u) * 1024);
  };

  f32x4 acc[MT][NW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int b = 0; b < NW; ++b) acc[i][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  if (n_it > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, d);
    int slot = 0;
    for (int it = 0; it < n_it; ++it) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"((D - 1) * L) : "memory");
      const char* at = ring + slot * (L * 1024);
      f32x4 av[2][MT];
      float bv[2][4][NW];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
          av[h][m] = *reinterpret_cast<const f32x4*>(at + m * 2048 + c * 128 +
                                                     16 * ((4 * h + g) ^ (c >> 1)));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = 4 * i + g;
#pragma unroll
          for (int b = 0; b < NW; ++b)
            bv[h][i][b] = *reinterpret_cast<const float*>(
                at + (2 * MT + h * NW) * 1024 + p * (64 * NW) + 64 * (b ^ swz(p)) + 4 * c);
        }
      }
      // The slot is refilled once this wave's reads of it are done.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(it + D, slot);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int b = 0; b < NW; ++b)
              acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[h][m][i], bv[h][i][b], acc[m][b],
                                                               0, 0, 0);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    // No load may land in the rings once they hold the waves' sums.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  const int rem = K % kRowsChunk;
  if (rem && wave == chunks % kRowsWaves) {
    const int64_t k0 = static_cast<int64_t>(chunks) * kRowsChunk;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = 16 * (i / 4) + 4 * g + i % 4;
      const bool in = k < rem;
      float av[MT], bv[NW];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = 16 * m + c < last ? 16 * m + c : last;
        av[m] = in ? A[static_cast<int64_t>(row) * K + k0 + k] : 0.0f;
      }
#pragma unroll
      for (int b = 0; b < NW; ++b) bv[b] = in ? B[(k0 + k) * N + n0 + 16 * b + c] : 0.0f;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int b = 0; b < NW; ++b)
          acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[m], bv[b], acc[m][b], 0, 0, 0);
    }
  }

  // Sums in wave order.  Lane (g, c), register r of block (m, b): row 16 m + 4 g + r,
  // column 16 b + c.
  __syncthreads();
  float* sums = reinterpret_cast<float*>(smem);
  constexpr int kOut = MT * NW * 256;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int b = 0; b < NW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sums[wave * kOut + ((m * NW + b) * 4 + r) * 64 + lane] = acc[m][b][r];
  __syncthreads();
  for (int o = threadIdx.x; o < kOut; o += kRowsThreads) {
    const int blk = o / 256, r = (o / 64) % 4, l = o % 64;
    const int row = m0 + 16 * (blk / NW) + 4 * (l / 16) + r;
    const int col = n0 + 16 * (blk % NW) + l % 16;
    if (row >= M || col < n_first) continue;
    float s = sums[o];
#pragma unroll
    for (int w = 1; w < kRowsWaves; ++w) s += sums[w * kOut + o];
    float* p = C + static_cast<int64_t>(row) * N + col;
    float v = alpha * s;
    if constexpr (FUSED) {
      const float bias = epi.bias[col];
      switch (epi.act) {
        case kActNone: v = epi_act<kActNone>(v, bias); break;
        case kActRelu: v = epi_act<kActRelu>(v, bias); break;
        case kActGeluErf: v = epi_act<kActGeluErf>(v, bias); break;
        default: v = epi_act<kActGeluTanh>(v, bias); break;
      }
    } else if (beta != 0.0f) {
      v += beta * *p;
    }
    *p = v;
  }
}

}  // namespace mcke_amd
