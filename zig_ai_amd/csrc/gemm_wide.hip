// The gated bfloat16 product of a step of many rows in the tiles of tiles_wide.h:
//
//   y [M, N] = act(x [M, K] . Wg [N, K]^T) * (x . Wu [N, K]^T),   W = [gate rows; up rows]
//
// A tile's weight rows are gate and up rows in turn, 16 each, so that a wave holds both columns and the
// products' 2N columns are neither written nor read again (a library's product and a kernel for the unit
// write and read them).  Full tiles of 256 rows and, at the end, one as low as holds what is left, 128, 192
// or 256: 1,037 rows make 4.5 rows of tiles.  Which products take it is the caller's rule.
// Measured (us; weights from memory, the library's product and the unit's kernel in brackets): 2 x 8192 x 2048
// at 2,048 rows 109 (123), 1.26 PFLOP/s; 2 x 7168 x 2048 at 1,037 60 (78), at 917 52 (60); 2 x 4608 x 1024 at
// 1,777 32 (42).  Without a unit the same tiles gain nothing: 6144 x 2048 at 2,048 rows 44 (42).
#include <type_traits>

#include "gate_unit.h"
#include "tiles_wide.h"

struct WideArgs {
  const bf16_t* x;
  const bf16_t* W;
  bf16_t* out;
  int M, N, K;
  float bound, slope, offset;
};

// UNIT: the unit's kind (gate_unit.h); ROUNDED: it reads the sums rounded to bfloat16, as a kernel of its own would
template <int UNIT, bool ROUNDED>
__global__ void __launch_bounds__(256, 1)
gemm_bf16_wide_gated_kernel(WideArgs g) {
  __shared__ __attribute__((aligned(16))) char lds[GW_LDS];
  // Workgroups are dealt to the eight dies in turn: a die takes an eighth of the full tiles, the rows of a
  // stretch of outputs side by side (its weights are read from memory once), then an eighth of the lower ones.
  const int columns = (g.N + 127) / 128, die = blockIdx.x & 7;
  const int rest = g.M & 255, rows = (g.M >> 8) + (rest > 192);
  const int full = rows * columns, low = rest > 0 && rest <= 192 ? columns : 0;
  const int full_each = (full + 7) >> 3, low_each = (low + 7) >> 3;
  int at = blockIdx.x >> 3;
  auto serve = [&](auto tm, int m0, int column) {
    constexpr int TM = decltype(tm)::value;
    using Tiles = TilesWide<TM>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = column * 128, M = g.M, N = g.N;
    const int lrow = wave * 8 + (lane >> 3), piece = ((lane & 7) ^ (lane >> 3)) * 16;
    unsigned offa[Tiles::LA], offw[Tiles::LW];
#pragma unroll
    for (int i = 0; i < Tiles::LA; ++i)      // (rows beyond are not stored)
      offa[i] = (unsigned)min(m0 + lrow + 32 * i, M - 1) * (unsigned)(g.K * 2) + piece;
#pragma unroll
    for (int i = 0; i < Tiles::LW; ++i) {
      const int tr = lrow + 32 * i, n = min(n0 + (tr >> 5) * 16 + (tr & 15), N - 1);
      offw[i] = (unsigned)(n + (tr & 16 ? N : 0)) * (unsigned)(g.K * 2) + piece;
    }
    f32x4_t acc[TM][Tiles::TN];
    Tiles::run(lds, wave, lane, g.K, (const char*)g.x, (const char*)g.W, offa, offw, acc, []() {});
    __syncthreads();
    const int wm = m0 + (wave >> 1) * 16 * TM;
    wide_store<bf16_t, 64, TM>(
        lds, wave, lane, g.out, n0 + (wave & 1) * 64, N,
        [&](int i, int j) {
          f32x4_t v;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float a = acc[i][2 * j][r], b = acc[i][2 * j + 1][r];
            v[r] = gated_value<UNIT, false>(ROUNDED ? (float)(bf16_t)a : a, ROUNDED ? (float)(bf16_t)b : b, g.bound, g.slope,
                                            g.offset);
          }
          return v;
        },
        [&](int i, int r) { return wm + 16 * i + r < M ? wm + 16 * i + r : -1; });
  };
  if (at < full_each) {
    const int index = die * full_each + at;
    if (index < full) serve(std::integral_constant<int, 8>{}, index % rows * 256, index / rows);
    return;
  }
  at -= full_each;
  const int index = die * low_each + at;
  if (at >= low_each || index >= low) return;
  if (rest > 128) serve(std::integral_constant<int, 6>{}, rows * 256, index);
  else serve(std::integral_constant<int, 4>{}, rows * 256, index);
}

// `kind`: gate_unit.h.  K is a multiple of 64, x and W start on 16 bytes and hold less than 4 GB each.
extern "C" int za_gemm_bf16_wide_gated(const void* x, const void* W, void* out, int M, int N, int K, int kind,
                                       float bound, float slope, float offset, int rounded, hipStream_t stream) {
  if (M == 0) return 0;
  if (M < 0 || N <= 0 || K <= 0 || !x || !W || !out || kind < 1 || kind > 3) return ZA_ERR_ARG;
  if (K % GG_BK != 0 || ((uintptr_t)x | (uintptr_t)W) % 16 != 0 || (long long)M * K > 0x7fffffffLL ||
      2LL * N * K > 0x7fffffffLL)
    return ZA_ERR_UNSUPPORTED;
  const long long columns = (N + 127LL) / 128, rows = (M + 255LL) / 256;
  const long long blocks = (rows * columns + 7) / 8 * 8 + 8;      // (two kinds, each an eighth a die)
  if (blocks > 0x7fffffffLL) return ZA_ERR_ARG;
  const WideArgs g{(const bf16_t*)x, (const bf16_t*)W, (bf16_t*)out, M, N, K, bound, slope, offset};
#define ZA_GW(UNIT)                                                                                                     \
  {                                                                                                                     \
    if (rounded)                                                                                                        \
      hipLaunchKernelGGL((gemm_bf16_wide_gated_kernel<UNIT, true>), dim3((unsigned)blocks), dim3(256), 0, stream, g);   \
    else                                                                                                                \
      hipLaunchKernelGGL((gemm_bf16_wide_gated_kernel<UNIT, false>), dim3((unsigned)blocks), dim3(256), 0, stream, g);  \
  }
  if (kind == 1) ZA_GW(1)
  else if (kind == 2) ZA_GW(2)
  else ZA_GW(3)
#undef ZA_GW
  return za_launch_status();
}
