// The dense projections of gemm.hip in 32-bit throughout (weights, sums; activations of either
// type): kernels of gemm_f32.h.
#include "common.h"
#include "gemm_f32.h"

#include <type_traits>

// dtype codes: 0 = float32, 1 = bfloat16
// Which kernel a 32-bit product takes: the tile whose workgroups fill the 256 compute units,
// waves that share a workgroup's K where they would not.  Measured (us; the FMA kernel that was
// here before these: 266 on average over 370 rows of the 350M shape's products, 14 TFLOP/s):
//   rows x N x K           rows 16x16  32x32 by 4  32x64 by 4  64x64 by 2   32x64   64x64
//    16 x  3072 x 1024            6.8        10.6        15.8
//    96 x  1024 x 1024           10.5        10.8        16
//   200 x  1024 x 4608           75          38          61
//   370 x  1024 x 4608                       75          62                    90     138
//   512 x  2048 x 2048                                   56          49        56      66
//   370 x  3072 x 1024                       46          44                    39      49
//  1024 x  9216 x 1024                                              219       202     191 (101 TFLOP/s)
//    16 x 65536 x 1024           79                      70                    65; by 2: 58
template <typename TA, typename TC, bool VEC>
static int launch_f32(const TA* A, const float* W, const float* bias, TC* C, int M, int N, int K, int wide,
                      hipStream_t stream) {
  auto tiles = [](int n, int t) { return (n + t - 1) / t; };
#define ZA_F32_GRID(BM, BN)                                      \
  const int mt = tiles(M, BM), nt = tiles(N, BN);                \
  const long long blocks = (long long)mt * ((nt + 7) / 8 * 8);   \
  if (blocks > 0x7fffffffLL) return ZA_ERR_ARG;                  \
  const dim3 grid((unsigned)blocks);
#define ZA_F32_TILE(BM, BN, KG)                                                                           \
  {                                                                                                       \
    ZA_F32_GRID(BM, BN)                                                                                   \
    hipLaunchKernelGGL((gemm_f32_tile_kernel<TA, TC, BM, BN, KG, VEC>), grid, dim3(256 * KG), 0, stream,  \
                       A, W, bias, C, M, N, K, mt, nt, wide);                                             \
    return za_launch_status();                                                                            \
  }
#define ZA_F32_ROWS(NW)                                                                                   \
  {                                                                                                       \
    ZA_F32_GRID(16, 16)                                                                                   \
    hipLaunchKernelGGL((gemm_f32_rows_kernel<TA, TC, NW, VEC>), grid, dim3(64 * NW), 0, stream, A,  \
                       W, bias, C, M, N, K, mt, nt, wide);                                                \
    return za_launch_status();                                                                            \
  }
  const bool few = M <= 16 ? N <= 16384 : (long long)tiles(M, 16) * tiles(N, 16) <= 384;
  if constexpr (VEC && std::is_same<TA, float>::value && std::is_same<TC, float>::value) {
    if (few) {
      if (K >= 2048) ZA_F32_ROWS(16)
      ZA_F32_ROWS(8)
    }
    if (M <= 16) ZA_F32_TILE(32, 64, 2)
    const long long n32 = (long long)tiles(M, 32) * tiles(N, 32), n3264 = (long long)tiles(M, 32) * tiles(N, 64),
                    n64 = (long long)tiles(M, 64) * tiles(N, 64);
#define ZA_F32_ASYNC(BM, BN, NS)                                                                          \
  {                                                                                                       \
    ZA_F32_GRID(BM, BN)                                                                                   \
    hipLaunchKernelGGL((gemm_f32_async_kernel<TC, BM, BN, NS>), grid, dim3(256), 0, stream, A, W, bias,   \
                       C, M, N, K, mt, nt, wide);                                                         \
    return za_launch_status();                                                                            \
  }
    // K in whole steps: tiles through LDS without registers, the same sums, reads and requests between the
    // products.  Measured, weights of several layers in turn, the kernels before it (with groups of waves that
    // took a step's reads, its products and its barrier one after the other) and now: 448 x 9216 x 1024 84 and
    // 65 (130 TFLOP/s), 350 x 9216 x 1024 84 and 61, 448 x 3072 x 1024 39 and 28, 448 x 2048 x 1024 26 and
    // 20, 448 x 1024 x 1024 15 and 11.5, 448 x 1024 x 4608 54 and 42.
    // 64 x 64 where the compute units take a tile half as often (0.93 of two of 32 x 64: 448 x 9216 65 and 68,
    // 448 x 3072 34 and 28).  A tile's rows are reached by 32-bit offsets in bytes: 64 K x 4 of them.
    if (K % F32_BK == 0 && n32 > 256 && K < (1 << 24)) {
      if (((n64 + 255) / 256) * 186 <= ((n3264 + 255) / 256) * 100) ZA_F32_ASYNC(64, 64, 4)
      ZA_F32_ASYNC(32, 64, 4)
    }
#undef ZA_F32_ASYNC
    if (n32 <= 256) ZA_F32_TILE(32, 32, 4)
    if (n3264 <= 256) ZA_F32_TILE(32, 64, 4)
    if (n64 <= 256) ZA_F32_TILE(64, 64, 2)
    // by how often the compute units take a tile (the smaller one, half the work, at 1.15 of its time)
    if (((n64 + 255) / 256) * 200 <= ((n3264 + 255) / 256) * 115) ZA_F32_TILE(64, 64, 1)
    ZA_F32_TILE(32, 64, 1)
  } else {
    // (weights that a checkpoint holds in 32-bit in a bfloat16 run, and widths that are no
    // multiple of four: one kernel for few rows and one for many)
    if (few) ZA_F32_ROWS(8)
    ZA_F32_TILE(32, 64, 2)
  }
#undef ZA_F32_TILE
#undef ZA_F32_ROWS
#undef ZA_F32_GRID
}

extern "C" int za_gemm_f32(const void* A, int a_dtype, const float* W, const float* bias, void* C,
                           int c_dtype, int M, int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  if (M < 0 || N < 0 || K <= 0 || !A || !W || !C) return ZA_ERR_ARG;
  const bool vec = K % 4 == 0 && (uintptr_t)A % (a_dtype == 1 ? 8 : 16) == 0 && (uintptr_t)W % 16 == 0;
  const int wide = N % 4 == 0 && (uintptr_t)C % 16 == 0;
#define ZA_F32_CASE(AD, TA, CD, TC)                                                                       \
  if (a_dtype == AD && c_dtype == CD)                                                                     \
    return vec ? launch_f32<TA, TC, true>((const TA*)A, W, bias, (TC*)C, M, N, K, wide, stream)           \
               : launch_f32<TA, TC, false>((const TA*)A, W, bias, (TC*)C, M, N, K, wide, stream);
  ZA_F32_CASE(0, float, 0, float)
  ZA_F32_CASE(1, bf16_t, 0, float)
  ZA_F32_CASE(1, bf16_t, 1, bf16_t)
  ZA_F32_CASE(0, float, 1, bf16_t)
#undef ZA_F32_CASE
  return ZA_ERR_UNSUPPORTED;
}
