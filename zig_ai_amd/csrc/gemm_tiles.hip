// bfloat16 matrix products of a step of 17 to 64 rows whose weights are what there is to read: a
// decode batch beyond the 16 rows of gemm_bf16_rows16.
//
//   y [M, N] = x [M, K] . W [N, K]^T,   M <= 64
//
// A workgroup takes 64 weight rows and one range of K, in tiles through LDS with all of the
// step's rows (tiles_bf16.h), three to five steps of 64 elements under way, so that it is bound by
// the weights' way from memory; the rows come from the die's cache each time.  Two workgroups
// share a compute unit; with few outputs K is cut into ranges until there are that many.
// Forms:
//   ranges   32-bit sums [ranges, M, N], K / ranges elements of K each (a multiple of 64)
//   plain    y in 32-bit or bfloat16
//   gated    W = [gate rows (N); up rows (N)], act(x . Wg^T) * (x . Wu^T) of the 32-bit sums in
//            bfloat16; a tile's weight rows are gate and up rows in turn, 16 each
// Measured (us; weights from memory, the library's product in brackets): gated 2 x 8192 x 2048
// 17.4 at 32 rows, 18.9 at 64 (with the kernel of the unit 20.9 and 21.1); 2048 x 8192 in 8 ranges
// 8.8 and 9.8 (10.4 and 13.8), 2048 x 2048 in 4 5.0 and 5.7 (6.0 and 6.6), 1024 x 4608 in 8 5.4 and
// 6.1 (8.4 and 8.5), 65536 x 2048 in 32-bit 58 and 64 (68 and 71).  Where a product without ranges
// leaves compute units idle the library stays: 6144 x 2048 11.5 and 12.8 (10.2 and 12.9).
#include "common.h"
#include "tiles_bf16.h"

#define GT_BN 64

// As the kernels for 16 rows have it: 0 silu, 1 gelu (tanh).
__device__ __forceinline__ float gt_unit(int act, float g, float u) {
  if (act == 0) return g / (1.0f + expf(-g)) * u;
  const float z = 0.7978845608028654f * (g + 0.044715f * g * g * g);
  return 0.5f * g * (1.0f + tanhf(z)) * u;
}

template <typename TO, bool GATED, int BM, int NS, bool ONCE>
__global__ void __launch_bounds__(256)
gemm_bf16_tiles_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, TO* __restrict__ out,
                       int M, int N, int K, int range, int act) {
  using Tiles = TilesBf16<BM, GT_BN, NS, ONCE>;
  __shared__ __attribute__((aligned(16))) bf16_t As[NS][BM * GG_BK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[NS][GT_BN * GG_BK];
  const int n0 = blockIdx.x * (GATED ? GT_BN / 2 : GT_BN), k0 = blockIdx.y * range;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lrow = wave * 8 + (lane >> 3), piece = (lane & 7) ^ (lane >> 3);
  const bf16_t* arow[Tiles::LA];
  const bf16_t* wrow[Tiles::LW];
#pragma unroll
  for (int i = 0; i < Tiles::LA; ++i)      // (rows beyond are not stored)
    arow[i] = x + (size_t)min(lrow + 32 * i, M - 1) * K + k0 + piece * 8;
#pragma unroll
  for (int i = 0; i < Tiles::LW; ++i) {
    const int tr = lrow + 32 * i;
    const int n = min(n0 + (GATED ? (tr >> 5) * 16 + (tr & 15) : tr), N - 1);
    wrow[i] = W + (size_t)(n + (GATED && (tr & 16) ? N : 0)) * K + k0 + piece * 8;
  }
  f32x4_t acc[Tiles::TM][Tiles::TN];
  Tiles::run(As, Ws, wave, lane, min(range, K - k0), arow, wrow, acc);
  const int wm = (wave % Tiles::WM) * (BM / Tiles::WM), wn = (wave / Tiles::WM) * (GT_BN / Tiles::WN);
  const int r16 = lane & 15, kq = lane >> 4;
  const bool wide = N % 4 == 0;            // (the launcher checks that `out` starts on 16 bytes)
#pragma unroll
  for (int i = 0; i < Tiles::TM; ++i) {
    const int row = wm + i * 16 + r16;
    if (row >= M) continue;
    TO* to = out + ((size_t)blockIdx.y * M + row) * N;
#pragma unroll
    for (int j = 0; j < Tiles::TN; j += GATED ? 2 : 1) {
      const int n = n0 + (GATED ? (wn >> 1) + (j / 2) * 16 : wn + j * 16) + kq * 4;
      if (n >= N) continue;
      f32x4_t v = acc[i][j];
      if constexpr (GATED) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = gt_unit(act, acc[i][j][r], acc[i][j + 1][r]);
      }
      if (wide) {
        if constexpr (sizeof(TO) == 4)
          *reinterpret_cast<f32x4_t*>(to + n) = v;
        else
          *reinterpret_cast<bf16x4_t*>(to + n) = bf16x4_t{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) to[n + r] = from_f32<TO>(v[r]);
      }
    }
  }
}

// out: [ranges][M][N] (bfloat16 only without ranges); `gated`: W is [2N][K], out bfloat16 [M][N].
// K is a multiple of 8, a range (all but the last of K / ranges rounded up to 64) not empty.
extern "C" int za_gemm_bf16_tiles(const void* x, const void* W, void* out, int out_dtype, int M, int N,
                                  int K, int ranges, int gated, int act, hipStream_t stream) {
  if (M == 0) return 0;
  if (M < 0 || M > 64 || N <= 0 || K <= 0 || ranges < 1 || ranges > 64 || !x || !W || !out || act < 0 || act > 1)
    return ZA_ERR_ARG;
  const int range = ((K + ranges - 1) / ranges + 63) / 64 * 64;
  if (K % 8 != 0 || (long long)(ranges - 1) * range >= K || (out_dtype != 0 && out_dtype != 1) ||
      (ranges > 1 && (gated || out_dtype != 0)) || (gated && out_dtype != 1) ||
      ((uintptr_t)x | (uintptr_t)W | (uintptr_t)out) % 16 != 0)
    return ZA_ERR_UNSUPPORTED;
  const int per = gated ? GT_BN / 2 : GT_BN;
  dim3 grid((unsigned)((N + per - 1) / per), (unsigned)ranges);
  // Large weights past the caches' other contents, by size: what comes from memory gains, what is left of the step
  // before in the last level's cache (256 MB) loses, and of weights of 32 MB and more a model of more than two or
  // three layers does not stay there.  Us as usual and past the caches, from memory and from the cache, 32 rows:
  // 8 MB 6.6 6.2 and 5.7 6.4, 17 MB 6.8 6.6 and 6.1 7.6, 25 MB 10.6 10.3 and 9.7 11.4, 34 MB 11.7 10.9 and
  // 10.1 12.9, 50 MB 14.1 12.3 and 11.3 14.3, 67 MB 17.4 15.3 and 14.3 17.5, 134 MB 30.1 27.8; 64 rows, 34 MB 13.2 12.9 and
  // 12.1 14.7, 67 MB 18.5 16.2 and 14.9 18.9.  In a decode step of 64 tokens of the 2,048-wide hybrid gate|up 18.6 and
  // 17.0, down 10.2 and 9.7, head 63.1 and 60.6, but 12 MB 9.5 and 9.7, 8 MB 5.6 and 5.8.
  const bool once = (gated ? 2LL : 1LL) * N * K * 2 >= ZA_ONCE_BYTES;
#define ZA_GT(TO, GATED, BM, NS)                                                                      \
  {                                                                                                   \
    if (once)                                                                                         \
      hipLaunchKernelGGL((gemm_bf16_tiles_kernel<TO, GATED, BM, NS, true>), grid, dim3(256), 0,       \
                         stream, (const bf16_t*)x, (const bf16_t*)W, (TO*)out, M, N, K, range, act);  \
    else                                                                                              \
      hipLaunchKernelGGL((gemm_bf16_tiles_kernel<TO, GATED, BM, NS, false>), grid, dim3(256), 0,      \
                         stream, (const bf16_t*)x, (const bf16_t*)W, (TO*)out, M, N, K, range, act);  \
  }
  // (65536 x 2048, 64 rows: 63.8 us with five places in LDS, 67.6 with four; in ranges four
  // are as good or better: 9.8 against 10.0)
  if (M <= 32) {
    if (gated) ZA_GT(bf16_t, true, 32, 6)
    else if (out_dtype == 0) ZA_GT(float, false, 32, 6)
    else ZA_GT(bf16_t, false, 32, 6)
  } else {
    if (gated) ZA_GT(bf16_t, true, 64, 4)
    else if (ranges > 1) ZA_GT(float, false, 64, 4)
    else if (out_dtype == 0) ZA_GT(float, false, 64, 5)
    else ZA_GT(bf16_t, false, 64, 5)
  }
#undef ZA_GT
  return za_launch_status();
}
