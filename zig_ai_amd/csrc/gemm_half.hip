// bfloat16 matrix products of a step of many rows whose outputs make one round of the tiles of tiles_half.h:
//
//   y [M, N] = x [M, K] . W [N, K]^T             in bfloat16
//   y [ranges, M, N]                             K in ranges of whole steps of 64, 32-bit sums that the reader
//                                                adds up
//
// Tiles of 256 x 256 leave most compute units idle there (1,037 rows and 3,072 outputs make 60 of them); these
// are as high as lets them fill one round.  Which products take it, with what height and how many ranges, is the
// caller's rule.  Measured (us; weights from memory, the library's product in brackets): 3072 x 2048 at 1,037
// rows 16.3 (20.2), 6144 x 2048 28.1 (29.7), 2048 x 2048 15.3 (16.3), at 2,048 rows 18.5 (20.8); in two ranges
// 2048 x 7168 at 1,037 rows 36 (added to the stream by the library 50), 2048 x 8192 at 2,048 rows 57 (68).
#include <type_traits>

#include "tiles_half.h"

struct HalfArgs {
  const bf16_t* x;
  const bf16_t* W;
  void* out;
  int M, N, K, range, ranges;
};

template <int TM, typename TO>
__global__ void __launch_bounds__(256, 1)
gemm_bf16_half_kernel(HalfArgs g) {
  using Tiles = TilesHalf<TM>;
  __shared__ __attribute__((aligned(16))) char lds[GW_LDS];
  // Workgroups are dealt to the eight dies in turn: a die takes an eighth of the tiles, the rows of a stretch of
  // outputs side by side (its weights are read from memory once).
  const int columns = (g.N + 127) / 128, rows = (g.M + 32 * TM - 1) / (32 * TM), total = rows * columns * g.ranges;
  const int each = (total + 7) >> 3, at = blockIdx.x >> 3, index = (blockIdx.x & 7) * each + at;
  if (at >= each || index >= total) return;
  const int stretch = index / rows, range = stretch / columns;
  const int m0 = (index - stretch * rows) * 32 * TM, n0 = (stretch - range * columns) * 128, M = g.M, N = g.N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = wave * 8 + (lane >> 3), piece = ((lane & 7) ^ (lane >> 3)) * 16;
  unsigned off[Tiles::LA + Tiles::LW];
#pragma unroll
  for (int i = 0; i < Tiles::LA; ++i)      // (rows beyond are not stored)
    off[i] = (unsigned)min(m0 + lrow + 32 * i, M - 1) * (unsigned)(g.K * 2) + piece;
#pragma unroll
  for (int i = 0; i < Tiles::LW; ++i)
    off[TM + i] = (unsigned)min(n0 + lrow + 32 * i, N - 1) * (unsigned)(g.K * 2) + piece;
  f32x4_t acc[TM][Tiles::TN];
  const int k0 = range * g.range;
  Tiles::run(lds, wave, lane, min(g.range, g.K - k0), (const char*)(g.x + k0), (const char*)(g.W + k0), off, acc);
  if (sizeof(TO) == 2) __syncthreads();
  const int wm = m0 + (wave >> 1) * 16 * TM;
  wide_store<TO, 64, TM>(
      lds, wave, lane, (TO*)g.out + (size_t)range * M * N, n0 + (wave & 1) * 64, N,
      [&](int i, int j) { return acc[i][j]; }, [&](int i, int r) { return wm + 16 * i + r < M ? wm + 16 * i + r : -1; });
}

// `height`: a tile's rows, 256, 192 or 128.  out_dtype 1: bfloat16 [M][N]; 0: 32-bit [ranges][M][N].  K is a multiple
// of 64; a range, all but the last of K / ranges rounded up to 64, is at least 320.  x and W start on 16 bytes and
// hold less than 4 GB each.
extern "C" int za_gemm_bf16_half(const void* x, const void* W, void* out, int out_dtype, int M, int N, int K,
                                 int height, int ranges, hipStream_t stream) {
  if (M == 0) return 0;
  if (M < 0 || N <= 0 || K <= 0 || ranges < 1 || !x || !W || !out) return ZA_ERR_ARG;
  if (K % GG_BK != 0 || (height != 256 && height != 192 && height != 128) || (out_dtype != 0 && out_dtype != 1) ||
      (ranges > 1 && out_dtype != 0) || ((uintptr_t)x | (uintptr_t)W) % 16 != 0 || (long long)M * K > 0x7fffffffLL ||
      (long long)N * K > 0x7fffffffLL || ranges > K / GG_BK)
    return ZA_ERR_UNSUPPORTED;
  const int range = (K / GG_BK + ranges - 1) / ranges * GG_BK;
  if (range < 5 * GG_BK || (long long)K - (long long)(ranges - 1) * range < 5 * GG_BK) return ZA_ERR_UNSUPPORTED;
  const long long tiles = (M + height - 1LL) / height * ((N + 127LL) / 128) * ranges, blocks = (tiles + 7) / 8 * 8;
  if (blocks > 0x7fffffffLL) return ZA_ERR_ARG;
  const HalfArgs g{(const bf16_t*)x, (const bf16_t*)W, out, M, N, K, range, ranges};
#define ZA_GH(TM)                                                                                                      \
  {                                                                                                                    \
    if (out_dtype == 1)                                                                                                \
      hipLaunchKernelGGL((gemm_bf16_half_kernel<TM, bf16_t>), dim3((unsigned)blocks), dim3(256), 0, stream, g);        \
    else                                                                                                               \
      hipLaunchKernelGGL((gemm_bf16_half_kernel<TM, float>), dim3((unsigned)blocks), dim3(256), 0, stream, g);         \
  }
  if (height == 256) ZA_GH(8)
  else if (height == 192) ZA_GH(6)
  else ZA_GH(4)
#undef ZA_GH
  return za_launch_status();
}
