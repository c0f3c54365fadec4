// A feed-forward of many small experts of which each token uses a few: the lists of
// who goes where, and products of every expert's rows with that expert's weights in one
// launch ("grouped" products).
//
// A step has A = T * top assignments; assignment a = t * top + j is token t's j-th expert.
//
// 1. expert_lists: one workgroup an expert walks the assignments in order and writes the
//    ones that name it, ascending, into lists[e][0 .. counts[e]).  No atomics, nothing to
//    clear beforehand, and the lists do not depend on the order in which anything ran.
//    Where an expert comes from is the caller's business: here a table indexed by the
//    token id, [vocab][top] (a router's top-k output [T][top] takes the same kernel with
//    the row index in place of the token id).
//
// 2. grouped_gemm: for every expert e and every tile of TM of its assignments,
//        out[dst(a)] = f(src[a / src_div] @ W[e]^T) * out_scale
//    src_div = top reads the tokens' rows, src_div = 1 rows that are already one an
//    assignment.  dst(a) = a, or, `stacked`, (a % top) * T + a / top: a stack [top][T][N]
//    of 32-bit partial results, which the norm that follows adds up in its order (so the
//    weighted sum over a token's experts is taken in 32-bit and costs no kernel).
//    f: nothing, or the square of relu; or, `gate`, the gated unit of two columns: W then has
//    2N rows, gate rows ahead of up rows, and out[.., n] = act(v[n]) * v[N + n] from the 32-bit
//    sums (a wave holds both columns), so the products' 2N columns are never stored.
//    `row_weight`: one number an assignment, times the result, or with a gate times the sums
//    ahead of it (a weight on an expert's input; there are no biases).  `rounded`: a gate reads its
//    sums rounded to the result's type, as a kernel of its own would.
//    How many tiles there are is known on the device only; the grid is the upper bound
//    ceil(A / TM) + E and a workgroup beyond the last tile leaves at once.
//    Every output element is a sum over k in an order fixed by K alone: a token's result
//    does not depend on which other tokens share its expert or its tile.
//      bfloat16: matrix cores (v_mfma_f32_16x16x32_bf16), tiles through LDS.
//      32-bit: tiles of 32 x 64 on the matrix cores' 32-bit instruction (gemm_f32.h).
#include <cmath>
#include <type_traits>

#include "common.h"
#include "gate_unit.h"
#include "gemm_f32.h"
#include "tiles_bf16.h"
#include "tiles_wide.h"

#define EX_MAX_EXPERTS 1024

// lists: int [E][A]; counts: int [E].  `ids` names the table's row for each token (null:
// the token's own index); an id outside [0, rows) names no expert.
// A workgroup an expert, which reads all assignments once: a thread takes up to EL_KEEP neighbouring
// ones, keeps as bits which of them name the expert, and writes those where they belong when the
// workgroup has added up the counts.  (A walk of 256 assignments at a time with a barrier each took
// 18.4 us for 7,108 assignments of 32 experts, all of it waiting.)
#define EL_KEEP 32
__global__ void __launch_bounds__(1024)
expert_lists_kernel(const int* __restrict__ ids, const int* __restrict__ table, int rows, int T,
                    int top, int* __restrict__ lists, int* __restrict__ counts) {
  __shared__ int wave_total[16];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int A = T * top;
  int* mine = lists + (size_t)e * A;
  const int span = min((A + (int)blockDim.x - 1) / (int)blockDim.x, EL_KEEP);
  int running = 0;
  for (long long base = 0; base < A; base += (long long)span * blockDim.x) {
    const long long first = base + (long long)tid * span;
    unsigned hits = 0;
#pragma unroll 8
    for (int i = 0; i < span; ++i) {
      const int a = (int)(first + i);
      bool hit = false;
      if (first + i < A) {
        const int t = a / top, id = ids ? ids[t] : t;
        hit = id >= 0 && id < rows && table[(size_t)id * top + (a - t * top)] == e;
      }
      hits |= (hit ? 1u : 0u) << i;
    }
    const int own = __popc(hits);
    int before = own;                     // over the wave, then over the waves
#pragma unroll
    for (int o = 1; o < ZA_WAVE; o <<= 1) {
      const int v = __shfl_up(before, o, ZA_WAVE);
      if (lane >= o) before += v;
    }
    __syncthreads();                      // the totals of the stretch before have been read
    if (lane == 63) wave_total[wave] = before;
    __syncthreads();
    int at = running + before - own;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
      if (w < wave) at += wave_total[w];
      running += wave_total[w];
    }
    for (unsigned left = hits; left; left &= left - 1) mine[at++] = (int)first + __ffs(left) - 1;
  }
  if (tid == 0) counts[e] = running;
}

extern "C" int za_expert_lists(const int* ids, const int* table, int rows, int n_tokens, int top,
                               int experts, int* lists, int* counts, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || top <= 0 || experts <= 0 || rows <= 0 || !table || !lists || !counts)
    return ZA_ERR_ARG;
  if (experts > EX_MAX_EXPERTS) return ZA_ERR_UNSUPPORTED;
  // (a workgroup of one wave for a decode batch, sixteen for long portions)
  const long long A = (long long)n_tokens * top;
  const int block = A <= 256 ? 64 : A <= 1024 ? 256 : 1024;
  hipLaunchKernelGGL(expert_lists_kernel, dim3(experts), dim3(block), 0, stream, ids, table, rows,
                     n_tokens, top, lists, counts);
  return za_launch_status();
}

struct GroupedArgs {
  const void* src;       // [rows][K]
  const void* W;         // [E][N][K]
  const int* lists;      // [E][A]
  const int* counts;     // [E]
  void* out;
  int A, T, top, E, N, K;
  int src_div, stacked, act;
  float out_scale;
  const float* row_weight;   // [A] or null
  int gate;                  // 0: none, 1: silu, 2: the tanh form of gelu, 3: bounded
  float bound, slope, offset;
  int rounded;               // with a gate: the sums are rounded to the result's type ahead of it
  unsigned per_magic;        // a / top, a < 2^31, as the upper half of a * per_magic, shifted (top > 1)
  int per_shift;
};

// The division of an assignment by `top`: a 32-bit division takes some 30 instructions, and a wide tile's rows
// have sixteen of them ahead of its first request.
__device__ __forceinline__ int token_of(const GroupedArgs& g, int a) {
  return g.top == 1 ? a : (int)(__umulhi((unsigned)a, g.per_magic) >> g.per_shift);
}

// The expert and the tile within it that workgroup `b` serves; false when there is none.  A wave
// looks at 64 experts at a time (every wave of the workgroup for itself; the answer is the same
// in all lanes).
template <int TM>
__device__ __forceinline__ bool find_tile(const int* __restrict__ counts, int E, int b, int* e_out,
                                          int* tile_out, int* count_out) {
  const int lane = threadIdx.x & 63;
  int first = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int c = e0 + lane < E ? counts[e0 + lane] : 0;
    const int tiles = (c + TM - 1) / TM;
    int end = tiles;                      // of the experts up to and including this lane's
#pragma unroll
    for (int o = 1; o < ZA_WAVE; o <<= 1) {
      const int v = __shfl_up(end, o, ZA_WAVE);
      if (lane >= o) end += v;
    }
    const unsigned long long past = __ballot(b < first + end);
    if (past) {
      const int at = __ffsll(past) - 1;
      *e_out = __builtin_amdgcn_readfirstlane(e0 + at);
      *count_out = __builtin_amdgcn_readlane(c, at);
      *tile_out = b - first - (__builtin_amdgcn_readlane(end, at) - __builtin_amdgcn_readlane(tiles, at));
      return true;
    }
    first += __builtin_amdgcn_readlane(end, 63);
  }
  return false;
}

// The number of tiles of all experts.
template <int TM>
__device__ __forceinline__ int count_tiles(const int* __restrict__ counts, int E) {
  int tiles = 0;
  for (int e = threadIdx.x & 63; e < E; e += 64) tiles += (counts[e] + TM - 1) / TM;
#pragma unroll
  for (int o = ZA_WAVE / 2; o > 0; o >>= 1) tiles += __shfl_xor(tiles, o, ZA_WAVE);
  return __builtin_amdgcn_readfirstlane(tiles);
}

__device__ __forceinline__ float expert_act(float v, int act) {
  if (act == 1) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return v;
}

// The gated unit (gate > 0) of one assignment's sums `v` (gate) and `u` (up).
template <typename TO, int KIND>
__device__ __forceinline__ float expert_unit(const GroupedArgs& g, bool rounded, float v, float u, float w) {
  constexpr bool EXACT = sizeof(TO) == 4;
  if constexpr (!EXACT) {
    const float rv = to_f32<TO>(from_f32<TO>(v)), ru = to_f32<TO>(from_f32<TO>(u));
    v = rounded ? rv : v;
    u = rounded ? ru : u;
  }
  return gated_value<KIND, EXACT>(v * w, u * w, g.bound, g.slope, g.offset);
}

// `what(kind)` with the unit's kind as a constant.
template <typename What>
__device__ __forceinline__ void with_unit(const GroupedArgs& g, What what) {
  if (g.gate == 1) what(std::integral_constant<int, 1>{});
  else if (g.gate == 2) what(std::integral_constant<int, 2>{});
  else what(std::integral_constant<int, 3>{});
}

__device__ __forceinline__ size_t dst_row(const GroupedArgs& g, int a) {
  if (!g.stacked) return (size_t)a;
  const int t = token_of(g, a);
  return (size_t)(a - t * g.top) * g.T + t;
}

// A wave's sums, acc[i][j][r] of assignment m + 16 i + lane % 16 of the expert's list and weight row
// wn + 16 j + lane / 16 * 4 + r of the tile that begins at output n0, on their way out.  GATED: the
// tile's weight rows are gate and up rows in turn, 16 each.
template <typename TO, bool GATED, int TM, int TN>
__device__ __forceinline__ void grouped_store(const GroupedArgs& g, const int* __restrict__ mine, int count,
                                              int m, int n0, int wn, int lane, const f32x4_t (&acc)[TM][TN]) {
  const int r16 = lane & 15, kq = lane >> 4;
  TO* out = (TO*)g.out;
  const int N = g.N;
  const bool wide = N % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & (4 * sizeof(TO) - 1)) == 0;
  auto put = [&](TO* to, int n, const f32x4_t& v) {      // outputs n .. n + 3 of one row
    if (wide) {
      if (n >= N) return;
      if constexpr (sizeof(TO) == 4) {
        *reinterpret_cast<f32x4_t*>(to + n) = v;
      } else {
        *reinterpret_cast<bf16x4_t*>(to + n) = bf16x4_t{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) to[n + r] = from_f32<TO>(v[r]);
    }
  };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = m + i * 16 + r16;
    if (row >= count) continue;
    TO* to = out + dst_row(g, mine[row]) * N;
    const float w = g.row_weight ? g.row_weight[mine[row]] : 1.0f;
    if constexpr (GATED) {
      with_unit(g, [&](auto kind) {
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
          f32x4_t v;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = expert_unit<TO, decltype(kind)::value>(g, g.rounded, acc[i][j][r], acc[i][j + 1][r], w);
          put(to, n0 + (wn >> 1) + (j / 2) * 16 + kq * 4, v);
        }
      });
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        f32x4_t v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = expert_act(acc[i][j][r], g.act) * g.out_scale * w;
        put(to, n0 + wn + j * 16 + kq * 4, v);
      }
    }
  }
}

// Tiles of BM assignments x BN weight rows (tiles_bf16.h).
// GATED: a tile is BN / 2 outputs; its weight rows are gate and up rows in turn, 16 each.
template <typename TO, bool GATED, int BM, int BN, int NS, bool ONCE>
__global__ void __launch_bounds__(256, 2)
grouped_gemm_bf16_tiled_kernel(GroupedArgs g) {
  using Tiles = TilesBf16<BM, BN, NS, ONCE>;
  constexpr int WM = Tiles::WM, WN = Tiles::WN, TM = Tiles::TM, TN = Tiles::TN, LA = Tiles::LA, LW = Tiles::LW;
  __shared__ __attribute__((aligned(16))) bf16_t As[NS][BM * GG_BK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[NS][BN * GG_BK];
  int e, tile, count;
  // workgroups are dealt to the eight dies in turn: a die takes an eighth of all tiles and stretches
  // of outputs, a tile's stretches side by side, so that few tiles (a decode batch's experts) keep
  // every die busy: with an eighth of the tiles each, nine tiles took five dies twice, two tiles two.
  // Many tiles of few stretches: an eighth of the tiles a die, for one stretch after the other, whose weights
  // an expert's tiles then share (side by side and so, us: 32 experts, 4,000 tokens, 4 each, 160 x 1,024, two
  // stretches, 22.3 and 20.2; 128 experts, 900 tokens, 8 each, gated 768 x 2,048, twelve, 128 and 137).
  // Tiles of 32, which a decode batch has, leave the choice out: it costs 0.3.
  const int columns = (g.N + (GATED ? BN / 2 : BN) - 1) / (GATED ? BN / 2 : BN);
  const int tiles = count_tiles<BM>(g.counts, g.E), die = blockIdx.x & 7, at = blockIdx.x >> 3;
  int which, stretch;
  if (BM > 32 && tiles >= 64 && columns <= 4) {
    const int per_die = (tiles + 7) >> 3;
    which = die * per_die + at % per_die;
    stretch = at / per_die;
    if (which >= tiles || stretch >= columns) return;
  } else {
    // (Each die begins 21 tiles further into its eighth than the one before: experts are a power of two
    // apart, and eight dies that walk one each in step meet in few of memory's channels.  8 experts of
    // 4,096 over 2,048, 20 tokens, gate|up, in step and 1, 5, 9, 13, 21 tiles apart: 62.7, 61.5, 53.4,
    // 54.8, 54.8, 54.4 us; 40 tokens 61.9 and (21) 54.7; 32 experts of 1,024, 64 tokens, with the down
    // product 49.9 + 26.9 and 53.5 + 25.5 (9), 50.9 + 25.9 (21); the others measured alike.)
    const int total = tiles * columns, per_die = (total + 7) >> 3;
    if (at >= per_die) return;
    const int turned = at + die * 21 % per_die, index = die * per_die + (turned < per_die ? turned : turned - per_die);
    if (index >= total) return;
    which = index / columns;
    stretch = index - which * columns;
  }
  const int n0 = stretch * (GATED ? BN / 2 : BN);
  if (!find_tile<BM>(g.counts, g.E, which, &e, &tile, &count)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
  const int* mine = g.lists + (size_t)e * g.A;
  const int K = g.K, N = g.N;
  const bf16_t* wbase = (const bf16_t*)g.W + (size_t)e * (GATED ? 2 * N : N) * K;

  // this lane's rows and its piece of their 128 bytes: row 32 i + 8 wave + lane / 8 of the tile
  const int lrow = wave * 8 + (lane >> 3), piece = (lane & 7) ^ (lane >> 3);
  const bf16_t* arow[LA];
  const bf16_t* wrow[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = min(tile * BM + lrow + 32 * i, count - 1);      // (rows beyond are not stored)
    arow[i] = (const bf16_t*)g.src + (size_t)(mine[r] / g.src_div) * K + piece * 8;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int tr = lrow + 32 * i;
    const int n = min(n0 + (GATED ? (tr >> 5) * 16 + (tr & 15) : tr), N - 1);
    wrow[i] = wbase + (size_t)(n + (GATED && (tr & 16) ? N : 0)) * K + piece * 8;
  }
  f32x4_t acc[TM][TN];
  Tiles::run(As, Ws, wave, lane, K, arow, wrow, acc);
  grouped_store<TO, GATED>(g, mine, count, tile * BM + wm, n0, wn, lane, acc);
}

// How many tiles of class CLASS (their rows) an expert of `c` assignments makes.  HIGH 256: full tiles of 256,
// and what is left at its end in one of 128 where that holds it; HIGH 128: tiles of 128 only.  (Ends of 192 as a
// third kind take the experts' tiles apart: 32 experts, 1,029 tokens unevenly, 4 each, 71 us instead of 70, down
// 40 instead of 38.)
template <int HIGH, int CLASS>
__device__ __forceinline__ int wide_tiles(int c) {
  if (HIGH == 128) return CLASS == 128 ? (c + 127) / 128 : 0;
  const int full = (c + 127) >> 8;
  return CLASS == 256 ? full : c > full * 256;
}

// Sums over a wave's lanes up to and including each, without LDS (six shuffles take some 600 clocks of waiting).
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // from 1, 2, 4, 8 lanes below in sixteen
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // the second and fourth sixteen: the one before
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);      // the upper half: the lower
  return v;
}

// Tile `b` of a class: its expert, the first of its assignments and the expert's count.  `own` is the count
// of the lane's expert among the first 64.
template <int HIGH, int CLASS>
__device__ __forceinline__ void wide_find(const int* __restrict__ counts, int E, int own, int b, int* e_out,
                                          int* m0_out, int* count_out) {
  const int lane = threadIdx.x & 63;
  int first = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int c = e0 == 0 ? own : e0 + lane < E ? counts[e0 + lane] : 0;
    const int tiles = wide_tiles<HIGH, CLASS>(c), end = wave_scan(tiles);
    const unsigned long long past = __ballot(b < first + end);
    if (past) {
      const int at = __ffsll(past) - 1, n = __builtin_amdgcn_readlane(c, at);
      const int tile = b - first - (__builtin_amdgcn_readlane(end, at) - __builtin_amdgcn_readlane(tiles, at));
      *e_out = __builtin_amdgcn_readfirstlane(e0 + at);
      *count_out = n;
      *m0_out = HIGH != CLASS ? n & ~255 : tile * HIGH;
      return;
    }
    first += __builtin_amdgcn_readlane(end, 63);
  }
}

// Tiles of 256 or 128 x 256 (tiles_wide.h); HIGH as above.  UNIT: 0 without, else GATED as above with the
// unit's kind as a constant, 4: any (for 32-bit results; the three kinds' stores side by side cost registers).
// ROUNDED: as g.rounded says (a choice an element takes six instructions).
template <typename TO, int UNIT, int HIGH, bool ROUNDED>
__global__ void __launch_bounds__(256, 1)
grouped_gemm_bf16_wide_kernel(GroupedArgs g) {
  constexpr bool GATED = UNIT > 0;
  __shared__ __attribute__((aligned(16))) char lds[GW_LDS];
  // Workgroups are dealt to the eight dies in turn: a die takes an eighth of the high tiles, an expert's
  // stretches of outputs side by side, and then an eighth of the low ones, which take half as long and
  // fill the ends.
  const int columns = (g.N + (GATED ? 127 : 255)) / (GATED ? 128 : 256), die = blockIdx.x & 7;
  int n256 = 0, n128 = 0;
  const int lane64 = threadIdx.x & 63, first64 = lane64 < g.E ? g.counts[lane64] : 0;
  for (int e0 = 0; e0 < g.E; e0 += 64) {
    const int c = e0 == 0 ? first64 : e0 + lane64 < g.E ? g.counts[e0 + lane64] : 0;
    n256 += wide_tiles<HIGH, 256>(c);
    n128 += wide_tiles<HIGH, 128>(c);
  }
  int at = blockIdx.x >> 3, index = -1;
  auto mine_of = [&](int tiles) {      // whether this workgroup's tile is one of a kind
    const int total = __builtin_amdgcn_readlane(wave_scan(tiles), 63) * columns, each = (total + 7) >> 3;
    if (at >= each) {
      at -= each;
      return false;
    }
    index = die * each + at < total ? die * each + at : -1;
    return true;
  };
  int e, m0, count;
  auto serve = [&](auto tm) {
    constexpr int TM = decltype(tm)::value;
    using Tiles = TilesWide<TM>;
    const int n0 = (index % columns) * (GATED ? 128 : 256);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int* mine = g.lists + (size_t)e * g.A;
    const int K = g.K, N = g.N;
    const int lrow = wave * 8 + (lane >> 3), piece = ((lane & 7) ^ (lane >> 3)) * 16;
    unsigned offa[Tiles::LA], offw[Tiles::LW];
#pragma unroll
    for (int i = 0; i < Tiles::LA; ++i) {
      const int r = min(m0 + lrow + 32 * i, count - 1);      // (rows beyond are not stored)
      const int a = mine[r];
      offa[i] = (unsigned)(g.src_div == 1 ? a : token_of(g, a)) * (unsigned)(K * 2) + piece;
    }
#pragma unroll
    for (int i = 0; i < Tiles::LW; ++i) {
      const int tr = lrow + 32 * i;
      const int n = min(n0 + (GATED ? (tr >> 5) * 16 + (tr & 15) : tr), N - 1);
      offw[i] = (unsigned)(n + (GATED && (tr & 16) ? N : 0)) * (unsigned)(K * 2) + piece;
    }
    // this lane's rows of the sums: where they go, and their weights
    const int wm = m0 + (wave >> 1) * 16 * TM, r16 = lane & 15;
    int to[TM];
    float weight[TM];
    f32x4_t acc[TM][Tiles::TN];
    Tiles::run(lds, wave, lane, K, (const char*)g.src, (const char*)g.W + (size_t)e * (GATED ? 2 * N : N) * K * 2, offa,
               offw, acc, [&]() {
#pragma unroll
                 for (int i = 0; i < TM; ++i) {
                   const int row = wm + 16 * i + r16, a = row < count ? mine[row] : -1;
                   to[i] = a < 0 ? -1 : (int)dst_row(g, a);
                   weight[i] = g.row_weight && a >= 0 ? g.row_weight[a] : 1.0f;
                 }
               });
    if (sizeof(TO) == 2) __syncthreads();
    auto put = [&](auto value) {
      wide_store<TO, GATED ? 64 : 128, TM>(
          lds, wave, lane, (TO*)g.out, n0 + (wave & 1) * (GATED ? 64 : 128), N,
          [&](int i, int j) {
            f32x4_t v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = value(i, j, r);
            return v;
          },
          [&](int i, int r) { return sizeof(TO) == 4 ? to[i] : __shfl(to[i], r, ZA_WAVE); });
    };
    if constexpr (UNIT == 4)
      with_unit(g, [&](auto kind) {
        put([&](int i, int j, int r) {
          return expert_unit<TO, decltype(kind)::value>(g, false, acc[i][2 * j][r], acc[i][2 * j + 1][r], weight[i]);
        });
      });
    else if constexpr (GATED)
      put([&](int i, int j, int r) {
        return expert_unit<TO, UNIT>(g, ROUNDED, acc[i][2 * j][r], acc[i][2 * j + 1][r], weight[i]);
      });
    else
      put([&](int i, int j, int r) { return expert_act(acc[i][j][r], g.act) * g.out_scale * weight[i]; });
  };
  if constexpr (HIGH == 256) {
    if (mine_of(n256)) {
      if (index < 0) return;
      wide_find<HIGH, 256>(g.counts, g.E, first64, index / columns, &e, &m0, &count);
      serve(std::integral_constant<int, 8>{});
      return;
    }
  }
  if (mine_of(n128)) {
    if (index < 0) return;
    wide_find<HIGH, 128>(g.counts, g.E, first64, index / columns, &e, &m0, &count);
    serve(std::integral_constant<int, 4>{});
  }
}

// 32-bit weights (src of either type): tiles of 32 assignments x 64 weight rows, the sums in the
// order of gemm_f32.h.  GATED: a tile is 32 outputs, its weight rows gate and up rows in turn, 16
// each, so that a lane holds both columns.
#define GF_BM 32
#define GF_BN 64

// VEC: 0 an element at a time, 1 four, 2 (32-bit rows, K a multiple of 32) through LDS without registers.
template <typename TA, typename TO, bool GATED, int VEC>
__global__ void __launch_bounds__(VEC == 2 ? 256 : 512)
grouped_gemm_f32_kernel(GroupedArgs g) {
  int e, tile, count;
  if (!find_tile<GF_BM>(g.counts, g.E, blockIdx.x, &e, &tile, &count)) return;
  const int n0 = blockIdx.y * (GATED ? GF_BN / 2 : GF_BN), m0 = tile * GF_BM;
  const int* mine = g.lists + (size_t)e * g.A;
  const int K = g.K, N = g.N;
  const float* W = (const float*)g.W + (size_t)e * (GATED ? 2 * N : N) * K;
  TO* out = (TO*)g.out;
  auto a_row = [&](int r) {
    const int a = mine[min(m0 + r, count - 1)];
    return g.src_div == 1 ? a : token_of(g, a);
  };
  auto w_row = [&](int r) {
    const int n = min(n0 + (GATED ? (r >> 5) * 16 + (r & 15) : r), N - 1);
    return n + (GATED && (r & 16) ? N : 0);
  };
  auto store = [&](int r, int n, const f32x4_t(&v)[GF_BN / 32]) {
    if (m0 + r >= count) return;
    const int a = mine[m0 + r];
    TO* at = out + dst_row(g, a) * N;
    const float w = g.row_weight ? g.row_weight[a] : 1.0f;
    if constexpr (GATED) {
      const int first = n0 + (n >> 5) * 16 + (n & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (first + i < N) with_unit(g, [&](auto kind) {
          at[first + i] = from_f32<TO>(expert_unit<TO, decltype(kind)::value>(g, g.rounded, v[0][i], v[1][i], w));
        });
    } else {
#pragma unroll
      for (int j = 0; j < GF_BN / 32; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n0 + n + j * 16 + i < N)
            at[n0 + n + j * 16 + i] = from_f32<TO>(expert_act(v[j][i], g.act) * g.out_scale * w);
    }
  };
  if constexpr (VEC == 2)
    f32_tile_async<GF_BM, GF_BN, 4>(K, (const float*)g.src, W, [&](int r) { return (unsigned)a_row(r) * (unsigned)(K * 4); },
                                    [&](int r) { return (unsigned)w_row(r) * (unsigned)(K * 4); }, store);
  else
    f32_tile<TA, GF_BM, GF_BN, 2, VEC == 1>(K, [&](int r) { return (const TA*)g.src + (size_t)a_row(r) * K; },
                                            [&](int r) { return W + (size_t)w_row(r) * K; }, store);
}

// Whether a grouped product reads its weights past the caches' other contents: few rows an expert, and
// more bytes than layers of which some could stay in the last level's cache (256 MB) from one step to the
// next would read, counted for the experts that A assignments can name and for the down product (gate|up
// reads twice that, so that two such layers and a half fill the cache).  What a step reads again loses by
// it, what comes from memory gains less.  Us, gate|up and down of a layer, as usual and past the caches, first
// with 180 MB of layers' weights that stay in the cache, then from memory; MB of the down product:
//   32 experts of 1,024 over 2,048, 4 a token, one token, 17 MB       19.4 23.6    24.2 23.1
//      2 tokens, 34 MB; 4, 67 MB                                      24.1 26.8    27.6 25.2;  40.0 36.8
//      8 tokens, 134 MB; 64; 400                                      58.7 54.1;  85.9 76.4;  106.6 98.0
//   32 of 512 over 1,024, one token, 4 MB; 8 tokens, 34 MB            12.6 13.8    14.5 13.7;  21.4 20.0
//   60 of 704 over 2,048, 4 a token, one token, 12 MB; 3, 35 MB       17.3 19.9    20.3 19.5;  28.1 26.0
//   8 of 2,048 over 1,024, 2 a token, one token, 8 MB; 8, 34 MB       17.8 20.4    21.1 20.3;  30.6 28.7
//   8 of 4,096 over 2,048, 2 a token, one token, 34 MB; 20, 134 MB    35.3 39.8    39.9 37.4;  95.7 86.0
//   8 of 1,024 over 1,024, 2 a token, 8 tokens, 17 MB                 17.4 19.4    19.4 18.6
// So the smaller sets, which a small model keeps (and a loop over layers reads twice a step), are left in.
extern "C" int za_grouped_reads_once(long long A, int experts, int N, int K) {
  return A < 80LL * experts && (A < experts ? A : experts) * N * K * 2 >= ZA_ONCE_BYTES;
}

// dtype codes: 0 = float32, 1 = bfloat16.  `src` has `src_rows` rows of K elements; the
// lists name assignments below n_tokens * top, so src_rows >= n_tokens (src_div == top) or
// >= n_tokens * top (src_div == 1).  With `gate` (see GroupedArgs) W is [experts][2N][K].
extern "C" int za_grouped_gemm(const void* src, int src_dtype, long long src_rows, const void* W,
                               int w_dtype, const int* lists, const int* counts, void* out,
                               int out_dtype, int n_tokens, int top, int experts, int N, int K,
                               int src_div, int stacked, int act, float out_scale,
                               const float* row_weight, int gate, float bound, float slope,
                               float offset, int rounded, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || top <= 0 || experts <= 0 || N <= 0 || K <= 0 || !src || !W || !lists ||
      !counts || !out || (src_div != 1 && src_div != top) || act < 0 || act > 1 ||
      gate < 0 || gate > 3 || (gate && (act || out_scale != 1.0f)))
    return ZA_ERR_ARG;
  const long long A = (long long)n_tokens * top;
  if (src_rows < (src_div == 1 ? A : (long long)n_tokens) || A > 0x7fffffff) return ZA_ERR_ARG;
  if (experts > EX_MAX_EXPERTS) return ZA_ERR_UNSUPPORTED;
  if (stacked && out_dtype != 0) return ZA_ERR_UNSUPPORTED;
  GroupedArgs g{src, W, lists, counts, out, (int)A, n_tokens, top, experts, N, K,
                src_div, stacked, act, out_scale, row_weight, gate, bound, slope, offset, rounded, 0, 0};
  if (top > 1) {      // 2^(31 + bits) / top, rounded up, fits 32 bits and is exact for a below 2^31
    int bits = 1;
    while ((1LL << bits) < top) ++bits;
    g.per_magic = (unsigned)(((1ULL << (31 + bits)) + top - 1) / top);
    g.per_shift = bits - 1;
  }
  if (w_dtype == 1) {
    if (src_dtype != 1 || K % 8 != 0 || ((uintptr_t)src | (uintptr_t)W) % 16 != 0) return ZA_ERR_UNSUPPORTED;
    if (out_dtype != 0 && out_dtype != 1) return ZA_ERR_UNSUPPORTED;
    // Tiles as high as the experts have rows on average, and one step of K under way, or as many
    // as keep memory busy where a launch makes fewer workgroups than the chip has compute units or
    // a decode batch reads little else than weights.  Measured with the weights of six layers in
    // turn, so that they come from memory as in a step (us, gate|up of 32 experts of 1,024 over 2,048
    // and their down product, 4 a token, evenly spread; the kernels before these: tiles of 128
    // through registers from 128 rows an expert on, 64 and 16 rows straight from memory below):
    //   tokens            8          64         260         400         517        1777
    //   before          51 + 25   167 + 85    184 + 96   226 + 118   229 + 123   140 + 90
    //    32 x  64       39 + 18    60 + 30     64 + 34    72 + 42     80 + 48    180 + 108
    //    64 x 128       43 + 20    64 + 26     66 + 28    66 + 30     80 + 43    122 + 78
    //   128 x 128       46 + 23    67 + 30     71 + 32    73 + 34     74 + 35    105 + 61
    //   the same, two steps under way                     80 + 37     81 + 38    125 + 76
    // (1,777 tokens, the fullest expert with 664 instead of 249: 131 + 77.  Weights left in the last
    // level's cache by the launch before gain a tenth to a third on these.)  8 experts of 4,096, 2 a
    // token: down 47 -> 32 at 20 tokens, 220 -> 52 at 500 (two steps under way; 73 with one).
    // Many rows an expert and K in whole steps of 64: the wide tiles, 256 assignments high where some 176
    // of them or more come about, else 128 where some 150 do (half an expert's tile more than its rows
    // make on average; below that compute units idle).  Measured as above, up | down (us): 32 experts of
    // 1,024 over 2,048, 4 a token, unevenly taken as a trained router does it, 1,777 tokens 141 | 78 ->
    // 110 | 66, 1,029 tokens 102 | 56 -> 83 | 42, 862 tokens 101 | 54 -> 79 | 39, 4,096 tokens 231 | 135
    // -> 182 | 107; at 517 tokens (65 rows an expert) 73 | 36 against 84 | 38.  8 experts of 4,096, 2 a
    // token, 1,900 tokens: up 99 -> 64 (128 high 85), down, 128 high for want of tiles, 92 -> 75 (256
    // high 95); 500 tokens: up, 128 high, 56 -> 43, down stays (54 against 66).  The sums are the same
    // to the last bit.  With four waves of 128 x 128 in place of eight of 128 x 64, the unit of
    // gate_unit.h and bfloat16 stored in whole lines, before and after (us): 32 experts, gated, 1,777 tokens 93
    // and 84, unevenly taken 105 and 94, 4,096 tokens 169 and 156, unevenly 163 and 148; 8 experts of 4,096,
    // gated, 1,777 tokens 173 and 158; their down product at 4,096 tokens 153 and 145.  32-bit results of few
    // steps of K are bound by the 58 MB and more that they write: 2,048 x 1,024, 1,777 tokens unevenly 58 and
    // 57, 1,024 tokens 38.4 and 39.3, unevenly 36.3 and 36.2, 1,277 45 and 42, 4,096 104 and 104; 64 experts of 2,048 x
    // 1,408, 6 a token, 1,093 tokens 96.4 and 95.5, unevenly 77.1 and 77.4.  Low tiles take longer at all of these.
    // And only where the rounds that the tiles make, 256 of them at a time or 512 of the low ones, take no
    // longer (few steps of K, outputs that fill little of a wide tile, a wide round that is nearly empty
    // where the low tiles make whole ones): a round of 128 x 128, two to a compute unit, as K, of 128 x 256 as
    // 0.9 K + 400, of 256 x 256 as 1.2 K + 400, an expert's last tile of those half as long; fitted to 420
    // products of 300 to 64,000 rows, 64 to 8,192 outputs and 128 to 4,096 elements of K with eight waves (us, low
    // and wide; with four, over 450 products, the choice is 1.5 percent from the best of the three on average):
    // 32 experts, 4 a token, gated, 8,000 tokens, 64 x 2,048 38 and 67; 4,000 tokens, 192 x 2,048 41 and 70;
    // 8 experts, 2 a token, gated, 12,000 tokens, 320 x 2,048 79 and 112, 448 x 2,048 115 and 117, 640 x
    // 2,048 157 and 131; not gated, 640 x 2,048 76 and 96, 512 x 2,048 72 and 56.
    if (K % GG_BK == 0 && A >= 80LL * experts && src_rows * K <= 0x7fffffffLL && (gate ? 2LL : 1LL) * N * K <= 0x7fffffffLL) {
      const long long columns = (N + (gate ? 127 : 255)) / (gate ? 128 : 256);
      int high = (A / 256 + experts / 2) * columns >= 176 ? 256
                 : (A / 128 + experts / 2) * columns >= 150 ? 128 : 0;
      const double tiles128 = A / 128.0 + experts / 2.0, low_columns = (N + (gate ? 63 : 127)) / (gate ? 64 : 128);
      const double low = ceil(tiles128 * low_columns / 512 + 0.06) * K;
      const double wide = high == 256 ? ceil((A / 256.0 + experts / 4.0) * columns / 128) / 2 * (1.2 * K + 400)
                                      : ceil(tiles128 * columns / 256) * (0.9 * K + 400);
      if (wide > low) high = 0;
      // (an expert's full tiles and its last one, each kind an eighth a die)
      const long long tiles = (A + high - 1) / max(high, 1) + experts;
      const long long blocks = (tiles * columns + 7) / 8 * 8 + 8;
      if (high && blocks > 0x7fffffffLL) return ZA_ERR_ARG;
#define ZA_GWH(TO, UNIT, HIGH, ROUNDED)                                                                    \
  hipLaunchKernelGGL((grouped_gemm_bf16_wide_kernel<TO, UNIT, HIGH, ROUNDED>), dim3((unsigned)blocks),     \
                     dim3(256), 0, stream, g)
#define ZA_GW(TO, UNIT)                                                                                    \
  {                                                                                                        \
    constexpr bool CHOICE = UNIT > 0 && UNIT < 4;                                                          \
    if (high == 256 && CHOICE && rounded) ZA_GWH(TO, UNIT, 256, CHOICE);                                   \
    else if (high == 256) ZA_GWH(TO, UNIT, 256, false);                                                    \
    else if (CHOICE && rounded) ZA_GWH(TO, UNIT, 128, CHOICE);                                             \
    else ZA_GWH(TO, UNIT, 128, false);                                                                     \
    return za_launch_status();                                                                             \
  }
      if (high) {
        if (out_dtype == 0) { if (gate) ZA_GW(float, 4) else ZA_GW(float, 0) }
        else if (gate == 0) ZA_GW(bf16_t, 0)
        else if (gate == 1) ZA_GW(bf16_t, 1)
        else if (gate == 2) ZA_GW(bf16_t, 2)
        else ZA_GW(bf16_t, 3)
      }
#undef ZA_GWH
#undef ZA_GW
    }
    const int BM = A >= 40LL * experts ? 128 : A >= 24LL * experts ? 64 : 32, BN = BM == 32 ? 64 : 128;
    const int columns = gate ? BN / 2 : BN;
    const long long rows = (A + BM - 1) / BM + experts, blocks = (rows + 7) / 8 * 8 * ((N + columns - 1) / columns);
    if (blocks > 0x7fffffffLL) return ZA_ERR_ARG;
    const dim3 grid((unsigned)blocks);
    const bool once = za_grouped_reads_once(A, experts, N, K) != 0;
#define ZA_GT(TO, GATED, BM, BN, NS)                                                                                \
  {                                                                                                                 \
    if (once)                                                                                                       \
      hipLaunchKernelGGL((grouped_gemm_bf16_tiled_kernel<TO, GATED, BM, BN, NS, true>), grid, dim3(256), 0, stream, \
                         g);                                                                                        \
    else                                                                                                            \
      hipLaunchKernelGGL((grouped_gemm_bf16_tiled_kernel<TO, GATED, BM, BN, NS, false>), grid, dim3(256), 0,        \
                         stream, g);                                                                                \
  }
#define ZA_GT_ROWS(TO, GATED)                                      \
  {                                                                \
    if (BM == 128 && blocks <= 256) ZA_GT(TO, GATED, 128, 128, 3)  \
    else if (BM == 128) ZA_GT(TO, GATED, 128, 128, 2)              \
    else if (BM == 64) ZA_GT(TO, GATED, 64, 128, 3)                \
    else ZA_GT(TO, GATED, 32, 64, 4)                               \
  }
    if (out_dtype == 0) { if (gate) ZA_GT_ROWS(float, true) else ZA_GT_ROWS(float, false) }
    else { if (gate) ZA_GT_ROWS(bf16_t, true) else ZA_GT_ROWS(bf16_t, false) }
#undef ZA_GT_ROWS
#undef ZA_GT
    return za_launch_status();
  }
  if (w_dtype != 0) return ZA_ERR_UNSUPPORTED;
  const int columns = gate ? GF_BN / 2 : GF_BN;
  dim3 grid((unsigned)((A + GF_BM - 1) / GF_BM + experts), (unsigned)((N + columns - 1) / columns)), block(512);
  const bool vec = K % 4 == 0 && (uintptr_t)src % (src_dtype == 1 ? 8 : 16) == 0 && (uintptr_t)W % 16 == 0;
  const bool whole = vec && src_dtype == 0 && K % F32_BK == 0 && src_rows * K < (1LL << 30) &&
                     (gate ? 2LL : 1LL) * N * K < (1LL << 30);
#define ZA_GFV(TA, TO, GATED)                                                                              \
  {                                                                                                        \
    if constexpr (std::is_same<TA, float>::value) {                                                        \
      if (whole) {                                                                                         \
        hipLaunchKernelGGL((grouped_gemm_f32_kernel<TA, TO, GATED, 2>), grid, dim3(256), 0, stream, g);    \
        return za_launch_status();                                                                         \
      }                                                                                                    \
    }                                                                                                      \
    if (vec) hipLaunchKernelGGL((grouped_gemm_f32_kernel<TA, TO, GATED, 1>), grid, block, 0, stream, g);   \
    else hipLaunchKernelGGL((grouped_gemm_f32_kernel<TA, TO, GATED, 0>), grid, block, 0, stream, g);       \
  }
#define ZA_GF(TA, TO)                 \
  {                                   \
    if (gate) ZA_GFV(TA, TO, true)    \
    else ZA_GFV(TA, TO, false)        \
  }
  if (src_dtype == 0 && out_dtype == 0) ZA_GF(float, float)
  else if (src_dtype == 1 && out_dtype == 0) ZA_GF(bf16_t, float)
  else if (src_dtype == 1 && out_dtype == 1) ZA_GF(bf16_t, bf16_t)
  else if (src_dtype == 0 && out_dtype == 1) ZA_GF(float, bf16_t)
  else return ZA_ERR_UNSUPPORTED;
#undef ZA_GF
#undef ZA_GFV
  return za_launch_status();
}

// ------------------------------------------------------------------------ a router
// Which `top` of `n` router outputs every token uses, and with which weight.  One wave a
// token, everything in 32-bit:
//   s = softmax(z) over all n outputs (mode 0) or sigmoid(z) (mode 1)
//   c = s + correction          the choice score (correction may be absent)
//   the outputs form `groups` equal groups of neighbours; a group's score is its largest c,
//   and only outputs of the `keep` best groups can be chosen (the others count as minus
//   infinity); groups == 0: no such limit
//   chosen = the `top` outputs with the largest c, in descending order (of equal scores the
//   lower index first); weight = s[chosen] * scale, or, `renorm`, divided by the sum of
//   the chosen s first
// What an output beyond the experts that have weights means (an expert that hands its input
// on, say) is the business of whoever reads `chosen`.
#define RT_MAX 1024

__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
  for (int o = ZA_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o, ZA_WAVE);
    const int oi = __shfl_xor(i, o, ZA_WAVE);
    if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
  }
}

__global__ void __launch_bounds__(64)
route_topk_kernel(const float* __restrict__ z, int ld, const float* __restrict__ correction, int n,
                  int groups, int keep, int top, float scale, int mode, int renorm,
                  int* __restrict__ chosen, float* __restrict__ weight) {
  __shared__ float ss[RT_MAX], cs[RT_MAX], gs[RT_MAX];
  const int t = blockIdx.x, lane = threadIdx.x;
  const float* zr = z + (size_t)t * ld;
  if (mode == 0) {
    float mx = -INFINITY;
    for (int e = lane; e < n; e += 64) mx = fmaxf(mx, zr[e]);
    mx = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < n; e += 64) {
      const float p = expf(zr[e] - mx);
      ss[e] = p;
      sum += p;
    }
    sum = wave_sum(sum);
    const float inv = 1.0f / sum;
    for (int e = lane; e < n; e += 64) ss[e] *= inv;
  } else {
    for (int e = lane; e < n; e += 64) ss[e] = 1.0f / (1.0f + expf(-zr[e]));
  }
  for (int e = lane; e < n; e += 64) cs[e] = ss[e] + (correction ? correction[e] : 0.f);
  __builtin_amdgcn_wave_barrier();
  __syncthreads();
  if (groups > 1 && keep < groups) {
    const int per = n / groups;
    for (int g = lane; g < groups; g += 64) {
      float best = -INFINITY;
      for (int k = 0; k < per; ++k) best = fmaxf(best, cs[g * per + k]);
      gs[g] = best;
    }
    __syncthreads();
    // the `keep` best groups get the mark +inf; afterwards every other group is closed
    for (int r = 0; r < keep; ++r) {
      float v = -INFINITY;
      int at = 0x7fffffff;
      for (int g = lane; g < groups; g += 64) {
        const float x = gs[g];
        if (x != INFINITY && (x > v || (x == v && g < at))) { v = x; at = g; }
      }
      wave_argmax(v, at);
      __syncthreads();
      if (lane == 0 && at < groups) gs[at] = INFINITY;
      __syncthreads();
    }
    for (int e = lane; e < n; e += 64)
      if (gs[e / per] != INFINITY) cs[e] = -INFINITY;
    __syncthreads();
  }
  float total = 0.f;
  for (int j = 0; j < top; ++j) {
    float v = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < n; e += 64) {
      const float x = cs[e];
      // (a taken output holds NaN, which compares false)
      if (x > v || (x == v && e < at)) { v = x; at = e; }
    }
    wave_argmax(v, at);
    __syncthreads();
    if (at >= n) at = 0;      // nothing left to choose from: cannot happen with top <= open outputs
    const float s = ss[at];
    total += s;
    if (lane == 0) {
      chosen[(size_t)t * top + j] = at;
      weight[(size_t)t * top + j] = s;
      cs[at] = __builtin_nanf("");
    }
    __syncthreads();
  }
  const float f = renorm ? scale / (total + 1e-20f) : scale;   // (all scores may underflow)
  for (int j = lane; j < top; j += 64) weight[(size_t)t * top + j] *= f;
}

// The same for at most 64 outputs: a lane has one, in registers.  Everything over the wave runs on the
// vector unit's own lane patterns (through LDS, a maximum over the wave waits six times): a choice is a
// maximum and the first lane that holds it, a group's best a maximum over its lanes.
// Where nearly all outputs are chosen for many tokens a lane counts the outputs before its own instead
// (`count`): the rounds are as many as the choices, the broadcasts as the outputs, and with enough waves to
// hide the waits their number decides.  Rounds and counting (us): 16,384 tokens, 32 outputs, 4, 12, 16,
// 24 and 32 of them 8 and 16, 16 and 17, 20 and 18, 28 and 20, 35 and 22; 64 outputs, 24, 32, 64 28 and 30, 35 and
// 32, 67 and 40; 2,048 tokens, 64 outputs, 32, 48, 64 8 and 9, 10 and 10, 13 and 11; up to 64 tokens rounds always.
// `z`: this lane's output, `give(j, output, weight)`: a lane that has the j-th choice.
struct RouteRule {
  int n, groups, keep, top, mode, renorm;
  float scale;
  int count;
};

static inline RouteRule route_rule(int n_tokens, int n, int groups, int keep, int top, int mode, int renorm,
                                   float scale) {
  const bool count = 5 * top > 2 * n && (long long)n_tokens * top >= 98304;
  return RouteRule{n, groups, keep, top, mode, renorm, scale, count ? 1 : 0};
}

template <int CTRL>
__device__ __forceinline__ float lanes_moved(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
// over 2, 4, 8, 16 neighbouring lanes: their pairs, quads, halves of rows, rows
#define ZA_OVER_16(v, OP)                     \
  v = OP(v, lanes_moved<0xB1>(v));            \
  v = OP(v, lanes_moved<0x4E>(v));            \
  v = OP(v, lanes_moved<0x141>(v));           \
  v = OP(v, lanes_moved<0x140>(v))
__device__ __forceinline__ float add_f32(float a, float b) { return a + b; }
__device__ __forceinline__ float lanes_max(float v) {
  ZA_OVER_16(v, fmaxf);
  return fmaxf(fmaxf(lane_value(v, 0), lane_value(v, 16)), fmaxf(lane_value(v, 32), lane_value(v, 48)));
}
__device__ __forceinline__ float lanes_sum(float v) {
  ZA_OVER_16(v, add_f32);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

template <typename F>
__device__ __forceinline__ void route_wave(const RouteRule& q, float z, float add, int lane, F&& give) {
  const bool in = lane < q.n;
  const float zv = in ? z : -INFINITY;
  float s;
  if (q.mode == 0) {
    const float p = in ? expf(zv - lanes_max(zv)) : 0.f;
    s = p * (1.0f / lanes_sum(p));
  } else {
    s = 1.0f / (1.0f + expf(-zv));
  }
  float c = s + (in ? add : 0.f);
  if (q.groups > 1 && q.keep < q.groups) {
    const int per = q.n / q.groups, g = lane / per;
    // (the largest that compares: NaN is nobody's best)
    float best = in && c == c ? c : -INFINITY;
    if (per == 2 || per == 4 || per == 8 || per == 16) {
      best = fmaxf(best, lanes_moved<0xB1>(best));
      if (per > 2) best = fmaxf(best, lanes_moved<0x4E>(best));
      if (per > 4) best = fmaxf(best, lanes_moved<0x141>(best));
      if (per > 8) best = fmaxf(best, lanes_moved<0x140>(best));
    } else {
      const float own = best;
      best = -INFINITY;
      for (int o = 0; o < q.groups; ++o) {
        const float v = lanes_max(g == o ? own : -INFINITY);
        best = o == g ? v : best;
      }
    }
    // (a group whose best is infinite is open whatever the others are)
    int before = 0;
    for (int k = 0; k < q.groups; ++k) {
      const float v = lane_value(best, k * per);
      if (v != INFINITY && (v > best || (v == best && k < g))) ++before;
    }
    if (best != INFINITY && before >= q.keep) c = -INFINITY;
  }
  bool open = in && c == c;                           // NaN is not chosen
  float total = 0.f, share = 0.f;
  if (q.count) {
    int before = 0;
#pragma unroll 8
    for (int k = 0; k < q.n; ++k) {
      const float v = lane_value(c, k);
      if (v > c || (v == c && k < lane)) ++before;
    }
    const int usable = __popcll(__ballot(open));
    for (int j = 0; j < q.top; ++j) {
      const unsigned long long who = __ballot(open && before == j);
      total += lane_value(s, j < usable ? __ffsll((long long)who) - 1 : 0);
    }
    const float f = q.renorm ? q.scale / (total + 1e-20f) : q.scale;
    if (open && before < q.top) give(before, lane, s * f);
    if (lane >= usable && lane < q.top) give(lane, 0, lane_value(s, 0) * f);
    return;
  }
  int place = -1, output = 0;
  for (int j = 0; j < q.top; ++j) {
    const float m = lanes_max(open ? c : -INFINITY);
    const unsigned long long who = __ballot(open && c == m);
    // (nothing left to choose from: output 0)
    const int at = who ? __ffsll((long long)who) - 1 : 0;
    const float v = lane_value(s, at);
    total += v;
    if (lane == j) {
      place = j;
      output = at;
      share = v;
    }
    if (lane == at) open = false;
  }
  const float f = q.renorm ? q.scale / (total + 1e-20f) : q.scale;   // (all scores may underflow)
  if (place >= 0) give(place, output, share * f);
}

__global__ void __launch_bounds__(64)
route_topk_wave_kernel(const float* __restrict__ z, int ld, const float* __restrict__ correction, RouteRule q,
                       int* __restrict__ chosen, float* __restrict__ weight) {
  const int t = blockIdx.x, lane = threadIdx.x;
  const bool in = lane < q.n;
  route_wave(q, in ? z[(size_t)t * ld + lane] : 0.f, in && correction ? correction[lane] : 0.f, lane,
             [&](int j, int output, float w) {
               chosen[(size_t)t * q.top + j] = output;
               weight[(size_t)t * q.top + j] = w;
             });
}

// A router from its product to its choice in one kernel, for at most 64 outputs (and a few rows behind
// them, the shared expert's gate): a workgroup takes MT * 16 tokens and all NT * 16 weight rows, its
// sixteen waves a sixteenth of K each (64 elements in turn, matrix cores, 32-bit sums added up in the
// waves' order), then a wave chooses for a token.  Where one workgroup has all tokens it writes the
// experts' lists, too.  Bound by its chain, way to memory, sums, choice, not by bytes; what it replaces
// is three or four launches with such a chain each, a product of 8 to 36 outputs that leaves all but a
// few compute units idle among them.  Measured in steps (us): 8 tokens, 33 weight rows of 2,048 elements
// 11.2 with the lists, for a product of 4.7, a choice of 7.1 and lists of 4.1; 20 tokens, 8 rows 8.9
// for a product of 4 to 8, a choice of 4.5 and lists of 4.5; prompts of 512 and 2,048 tokens 10.1 for
// two of the three (their lists, 5 to 9, stay apart: an expert's workgroup reads all assignments).
struct RouteArgs {
  const bf16_t *x, *W;       // [T][K], [rows][K]
  const float *bias, *correction;
  float* logits;             // [T][rows] or null
  int* chosen;               // [T][top]
  float* weight;             // [T][top]
  int* lists;                // [experts][T * top] or null: no lists
  int* counts;
  int T, K, rows, experts;
  RouteRule q;
};

#define RL_WAVES 16

template <int NT, int MT>
__global__ void __launch_bounds__(RL_WAVES * 64)
route_linear_kernel(RouteArgs a) {
  constexpr int LD = NT * 16 + 4, UNROLL = NT * MT > 3 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float sums[RL_WAVES][MT * 16][LD];
  __shared__ int picked[MT * 16 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int t0 = blockIdx.x * MT * 16, K = a.K;
  const bf16_t *xr[MT], *wr[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xr[i] = a.x + (size_t)min(t0 + i * 16 + r16, a.T - 1) * K;
#pragma unroll
  for (int j = 0; j < NT; ++j) wr[j] = a.W + (size_t)min(j * 16 + r16, a.rows - 1) * K;
  // (asked for ahead of the product)
  const float add = a.correction && lane < a.q.n ? a.correction[lane] : 0.f;
  const float shift = a.bias ? a.bias[min(tid % (NT * 16), a.rows - 1)] : 0.f;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // (a wave reads whole lines of 128 bytes, 64 elements)
  for (int k0 = wave * 64 + kq * 8; k0 - kq * 8 < K; k0 += UNROLL / 2 * RL_WAVES * 64) {
    bf16x8_t fx[UNROLL][MT], fw[UNROLL][NT];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int k = k0 + (u >> 1) * RL_WAVES * 64 + (u & 1) * 32, at = min(k, K - 8);      // (K is a multiple of 8)
#pragma unroll
      for (int i = 0; i < MT; ++i) fx[u][i] = *reinterpret_cast<const bf16x8_t*>(xr[i] + at);
#pragma unroll
      for (int j = 0; j < NT; ++j) fw[u][j] = *reinterpret_cast<const bf16x8_t*>(wr[j] + at);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const bool in = k0 + (u >> 1) * RL_WAVES * 64 + (u & 1) * 32 < K;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(in ? fw[u][j] : zero8, in ? fx[u][i] : zero8,
                                                               acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *reinterpret_cast<f32x4_t*>(&sums[wave][i * 16 + r16][j * 16 + kq * 4]) = acc[i][j];
  __syncthreads();
  for (int i = tid; i < MT * 16 * NT * 16; i += RL_WAVES * 64) {
    const int t = i / (NT * 16), o = i % (NT * 16);
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < RL_WAVES; ++w) v += sums[w][t][o];
    if (a.bias && o < a.rows) v += i < RL_WAVES * 64 ? shift : a.bias[o];
    sums[0][t][o] = v;                               // (only this thread reads or writes the place)
    if (a.logits && o < a.rows && t0 + t < a.T) a.logits[(size_t)(t0 + t) * a.rows + o] = v;
  }
  __syncthreads();
  for (int i = 0; i < MT; ++i) {
    const int own = i * RL_WAVES + wave, t = t0 + own;
    if (t >= a.T) break;
    route_wave(a.q, lane < a.q.n ? sums[0][own][lane] : 0.f, add, lane, [&](int j, int output, float w) {
      a.chosen[(size_t)t * a.q.top + j] = output;
      a.weight[(size_t)t * a.q.top + j] = w;
      picked[own * a.q.top + j] = output;
    });
  }
  if (!a.lists) return;
  __syncthreads();
  const int A = a.T * a.q.top;
  for (int e = wave; e < a.experts; e += RL_WAVES) {
    int running = 0;
    for (int base = 0; base < A; base += 64) {
      const bool hit = base + lane < A && picked[base + lane] == e;
      const unsigned long long who = __ballot(hit);
      if (hit) a.lists[(size_t)e * A + running + __popcll(who & ((1ull << lane) - 1))] = base + lane;
      running += __popcll(who);
    }
    if (lane == 0) a.counts[e] = running;
  }
}

// `rows` weight rows, the first `n` of them the router's outputs; lists and counts may be null (they must
// be beyond ZA_ROUTE_LISTS tokens: no workgroup sees all of them).
#define ZA_ROUTE_LISTS 32
extern "C" int za_route_linear(const void* x, const void* W, const float* bias, const float* correction,
                               int n_tokens, int K, int rows, int n, int groups, int keep, int top, float scale,
                               int mode, int renorm, float* logits, int* chosen, float* weight, int experts,
                               int* lists, int* counts, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || K <= 0 || n <= 0 || rows < n || top <= 0 || top > n || !x || !W || !chosen || !weight ||
      groups < 0 || (groups > 0 && (n % groups != 0 || keep <= 0 || keep > groups)) || mode < 0 || mode > 1 ||
      (lists && (!counts || experts <= 0 || n_tokens > ZA_ROUTE_LISTS)))
    return ZA_ERR_ARG;
  if (groups > 0 && (long long)keep * (n / groups) < top) return ZA_ERR_ARG;
  if (n > 64 || rows > 80 || K % 8 != 0 || ((uintptr_t)x | (uintptr_t)W) % 16 != 0) return ZA_ERR_UNSUPPORTED;
  const int tiles = (rows + 15) / 16;
  const bool two = lists && n_tokens > 16;            // (all tokens in one workgroup)
  if (two && tiles > 3) return ZA_ERR_UNSUPPORTED;
  RouteArgs a{(const bf16_t*)x, (const bf16_t*)W, bias, correction, logits, chosen, weight, lists, counts,
              n_tokens, K, rows, experts, route_rule(n_tokens, n, groups, keep, top, mode, renorm, scale)};
  const dim3 grid(two ? 1 : (n_tokens + 15) / 16), block(RL_WAVES * 64);
#define ZA_RL(NT, MT) hipLaunchKernelGGL((route_linear_kernel<NT, MT>), grid, block, 0, stream, a)
  if (two) {
    if (tiles == 1) ZA_RL(1, 2);
    else if (tiles == 2) ZA_RL(2, 2);
    else ZA_RL(3, 2);
  } else if (tiles == 1) ZA_RL(1, 1);
  else if (tiles == 2) ZA_RL(2, 1);
  else if (tiles == 3) ZA_RL(3, 1);
  else if (tiles == 4) ZA_RL(4, 1);
  else ZA_RL(5, 1);
#undef ZA_RL
  return za_launch_status();
}

extern "C" int za_route_topk(const float* z, int ld, const float* correction, int n_tokens, int n,
                             int groups, int keep, int top, float scale, int mode, int renorm,
                             int* chosen, float* weight, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || n <= 0 || ld < n || top <= 0 || top > n || !z || !chosen || !weight ||
      groups < 0 || (groups > 0 && (n % groups != 0 || keep <= 0 || keep > groups)) ||
      mode < 0 || mode > 1)
    return ZA_ERR_ARG;
  if (groups > 0 && (long long)keep * (n / groups) < top) return ZA_ERR_ARG;
  if (n > RT_MAX) return ZA_ERR_UNSUPPORTED;
  if (n <= 64)
    hipLaunchKernelGGL(route_topk_wave_kernel, dim3(n_tokens), dim3(64), 0, stream, z, ld, correction,
                       route_rule(n_tokens, n, groups, keep, top, mode, renorm, scale), chosen, weight);
  else
    hipLaunchKernelGGL(route_topk_kernel, dim3(n_tokens), dim3(64), 0, stream, z, ld, correction, n,
                       groups, keep, top, scale, mode, renorm, chosen, weight);
  return za_launch_status();
}

// What a token's chosen experts and the shared expert give, as one 32-bit row:
//   y[t] = sum_j weight[t][j] * (chosen[t][j] < n_real ? expert_out[t * top + j] : x[t])
//          + gate(t) * shared[t]
// An output beyond the n_real experts that have weights hands the token's input x[t] on.
// gate(t) = sigmoid(gate_logits[t * gate_ld]) when gate_logits is given, else 1; `shared`
// may be absent.  The sum is taken in the order j = 0 .. top - 1, then the shared expert.
// With `stream` the row goes there, stream[t] += stream_scale * y[t], and rounded to `copy` (may be
// null); otherwise to y.
// `weigh` 0: the experts' outputs hold their weights already (a weight on an expert's input).
// A thread takes one column of one token (a workgroup 256 of them: with a workgroup a token and its
// columns one after the other, eight tokens of 2,048 took 14.9 us).
template <typename TE, typename TX, bool ADD>
__global__ void __launch_bounds__(256)
experts_combine_kernel(const TE* __restrict__ expert_out, const int* __restrict__ chosen,
                       const float* __restrict__ weight, const TX* __restrict__ x,
                       const TE* __restrict__ shared, const float* __restrict__ gate_logits,
                       int gate_ld, float* __restrict__ y, int top, int n_real, int width,
                       int weigh, float stream_scale, bf16_t* __restrict__ copy) {
  const size_t t = blockIdx.x;
  const int i = blockIdx.y * blockDim.x + threadIdx.x;
  if (i >= width) return;
  const float sh = shared ? to_f32<TE>(shared[t * width + i]) : 0.f;
  const float own = to_f32<TX>(x[t * width + i]);
  const float before = ADD ? y[t * width + i] : 0.f;
  float g = 1.0f;
  if (shared && gate_logits) g = 1.0f / (1.0f + expf(-gate_logits[t * gate_ld]));
  float acc = 0.f;
#pragma unroll 4
  for (int j = 0; j < top; ++j) {
    const int e = chosen[t * top + j];
    const float w = (weigh || e >= n_real) ? weight[t * top + j] : 1.f;
    const float v = e < n_real ? to_f32<TE>(expert_out[(t * top + j) * width + i]) : own;
    acc = fmaf(w, v, acc);
  }
  if (shared) acc = fmaf(g, sh, acc);
  if (ADD) acc = fmaf(stream_scale, acc, before);
  y[t * width + i] = acc;
  if (ADD && copy) copy[t * width + i] = (bf16_t)acc;
}

// dtype codes: 0 = float32, 1 = bfloat16; `out_dtype` is that of expert_out and shared.
extern "C" int za_experts_combine(const void* expert_out, int out_dtype, const int* chosen,
                                  const float* weight, const void* x, int x_dtype,
                                  const void* shared, const float* gate_logits, int gate_ld,
                                  float* y, int n_tokens, int top, int n_real, int width,
                                  int weigh, int add, float stream_scale, void* copy, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || top <= 0 || width <= 0 || n_real < 0 || !chosen || !weight || !x || !y ||
      (n_real > 0 && !expert_out) || (copy && !add))
    return ZA_ERR_ARG;
  dim3 block(width <= 256 ? 64 : 256), grid(n_tokens, (width + block.x - 1) / block.x);
#define ZA_ECA(TE, TX, ADD)                                                                    \
  hipLaunchKernelGGL((experts_combine_kernel<TE, TX, ADD>), grid, block, 0, stream,            \
                     (const TE*)expert_out, chosen, weight, (const TX*)x, (const TE*)shared,   \
                     gate_logits, gate_ld, y, top, n_real, width, weigh, stream_scale, (bf16_t*)copy)
#define ZA_EC(TE, TX)                   \
  {                                     \
    if (add) ZA_ECA(TE, TX, true);      \
    else ZA_ECA(TE, TX, false);         \
  }
  if (out_dtype == 0 && x_dtype == 0) ZA_EC(float, float)
  else if (out_dtype == 0 && x_dtype == 1) ZA_EC(float, bf16_t)
  else if (out_dtype == 1 && x_dtype == 1) ZA_EC(bf16_t, bf16_t)
  else if (out_dtype == 1 && x_dtype == 0) ZA_EC(bf16_t, float)
  else return ZA_ERR_UNSUPPORTED;
#undef ZA_EC
#undef ZA_ECA
  return za_launch_status();
}
