// Long portions through the mixers that carry a matrix state (recurrent.hip has their
// recurrences, their layouts and the token-by-token walk that decode batches take): chunks of
// tokens as matrix products on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32:
// products and sums in 32-bit).  Lane l = 16 g + r of it supplies row r and k element g of either
// operand and receives rows 4 g .. + 3 and column r of the product.  The order in which k runs is
// free as long as both operands agree: step j of a block of sixteen takes elements 4 g + j, so a
// lane's four steps are four neighbouring floats, and a product's own layout is that of an
// operand whose k runs along its rows.
#include <math.h>

#include "common.h"

__device__ __forceinline__ f32x4_t mfma4(const f32x4_t& a, const f32x4_t& b, f32x4_t c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  return c;
}

__device__ __forceinline__ f32x4_t zero4() { return f32x4_t{0.f, 0.f, 0.f, 0.f}; }

// Four consecutive floats, those at and beyond `n` as zeros.
__device__ __forceinline__ f32x4_t load4_below(const float* p, int n, bool aligned) {
  f32x4_t v = zero4();
  if (aligned && n >= 4) return *reinterpret_cast<const f32x4_t*>(p);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < n) v[j] = p[j];
  return v;
}

// The same without a condition where the kernel's caller has seen that all four are there (FULL): a
// load behind a condition is waited for where the two ways meet again.
template <bool FULL>
__device__ __forceinline__ f32x4_t load4(const float* p, int n, bool aligned) {
  if constexpr (FULL) return *reinterpret_cast<const f32x4_t*>(p);
  else return load4_below(p, n, aligned);
}

// Whether any lane holds a number that is infinite or none (zero times such a number is not zero).
__device__ __forceinline__ bool any_wild(const f32x4_t& v) {
  const float z = (v[0] * 0.f + v[1] * 0.f) + (v[2] * 0.f + v[3] * 0.f);
  return __any(z != 0.f);
}

__device__ __forceinline__ f32x4_t without_wild(const f32x4_t& v) {
  f32x4_t x;
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = v[j] * 0.f == 0.f ? v[j] : 0.f;
  return x;
}

// For a block of sixteen tokens that are their own keys (rows 4 g + j of v, as a second operand):
// from a wild number's row on every sum of its column in c is no number.  (A later token's weight
// of zero does not keep such a number out, so the product is taken without.)
__device__ __forceinline__ void wild_from_its_row(const f32x4_t& v, f32x4_t& c, int g) {
  int first = 16;
#pragma unroll
  for (int j = 3; j >= 0; --j)
    if (v[j] * 0.f != 0.f) first = 4 * g + j;
  first = min(first, __shfl_xor(first, 16, ZA_WAVE));
  first = min(first, __shfl_xor(first, 32, ZA_WAVE));
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g + r >= first) c[r] = __builtin_nanf("");
}

__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// ------------------------------------------------------------- one decay a head and token
// State-space duality and fixed decays:  S <- a S + dt k v^T,  o = S^T q (+ D v), with a one
// number a head, a function of the token or constant.  With c_i = log2 of the product of a chunk's
// decays up to and including token i (in double, kept as two floats: a difference of two of them
// is put together before the power is taken, so its error does not grow with the sum), n its
// tokens, B the state before it:
//   1. decay_chunk_state:   N = sum_j 2^(c_n - c_j) dt_j k_j v_j^T   of every chunk by itself
//   2. decay_prefix:        B of every chunk in a request's order, B <- 2^c_n B + N
//   3. decay_chunk_out:     o_i = 2^c_i B^T q_i + sum_(j <= i) 2^(c_i - c_j) dt_j (q_i . k_j) v_j
// Every factor is a power of at most zero while decays are at most one.  All products are matrix
// products of 16 x 16 x dk and 16 x 16 x dv blocks; the walk is a chain of tokens instead, 0.34 us
// each.  2,048 tokens, 64 heads of 128 x 64: 698 us walked; 33 + 16 + 51 + 7 us here, where the heads share
// their scores (a head's own take 15 us and most of the registers); 16 heads of 128 x 128:
// 624 us walked, 70 here (92 as chunks of 256 walked side by side and corrected).  The products' time is 14 + 21 us;
// all workgroups are on the chip at once and load, multiply and store at the same time, 67 + 67 + 100 MB in
// all.  Where the sizes are whole, tiles take neighbouring channels and columns a lane, so that rows are read
// and written 16 bytes at a time, and the state before a chunk goes into LDS once (element by element, a wave all
// key channels, and the state a wave: 44 and 64 in place of the 33 and 51).
#define DC_CHUNK 128

// Four neighbouring floats from any place on (memory takes 16 bytes a lane from any multiple of 4).
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any_t;

// The least log2 of a decay that is told apart from zero.  Any power this small is zero in 32-bit
// (2^-149 is the last that is not), and a chunk's sum of such numbers still has 37 binary places in
// double, so the decays behind a token that forgets everything keep theirs.
#define DC_LEAST_LOG2 -400.0

// 2^(hi + lo), |lo| at most a few last places of the sum that hi came from.
__device__ __forceinline__ float exp2_of(float hi, float lo) {
  const float e = hi + lo, rest = (hi - e) + lo;      // (rest: below the last place of e)
  return exp2f(e) * fmaf(rest, 0.6931471805599453f, 1.0f);
}

struct DecayArgs {
  const float* vec;        // [T][width]: q at q_col + g*dk, k at k_col + g*dk, v at x_col + h*dv
  int width, q_col, k_col, x_col;
  const void* proj;        // [T][proj_stride] storage type: the raw step size at gate_col + h
  int proj_stride, gate_col, proj_bf16;
  const float* dt_bias;    // [H]
  const float* A_log;      // [H]
  const float* D;          // [H], or null
  const float* fixed;      // [H] constant decays, or null (dt is one then)
  const int* item_row0;
  const int* item_count;
  float* sums;             // [T][H][3]: c as two floats, dt
  float* chunk_state;      // [items][H][dv][dk]
  float* total;            // [items][H]: 2^c_n
  float* out;              // [T][H*dv]
  int H, G, dk, dv;
  float* scores;           // [items][G][128][128]: q_i . k_j, j <= i to whole blocks of 16; or null
};

// One workgroup a chunk, head and 64 columns; a wave takes 16 columns.
// FULL: dk fills its tiles and dv its 64 columns.
template <int NT, bool FULL>      // tiles of 16 key channels
__global__ void __launch_bounds__(256)
decay_chunk_state_kernel(DecayArgs a) {
  __shared__ __attribute__((aligned(16))) float weight[DC_CHUNK];
  __shared__ double first_half, whole;
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4;
  const int row0 = a.item_row0[item], n = a.item_count[item];
  const int dk = a.dk, dv = a.dv;

  // FULL: a wave takes half of the key channels and 32 columns, neighbouring ones a lane, so that a key's are read 16
  // bytes at a time (8 at states of 64 rows) and a value's 8: tile t's row r is channel r * CT + t, tile c's column
  // 2 r + c.  Otherwise all key channels and 16 columns, an element at a time.
  constexpr int CT = FULL ? NT / 2 : NT, VT = FULL ? 2 : 1;      // tiles of channels, and of columns
  typedef __attribute__((ext_vector_type(CT))) float keys_t;
  typedef __attribute__((ext_vector_type(VT), aligned(4))) float values_t;      // (x_col may be any)
  const int chan0 = FULL ? (wave & 1) * CT * 16 : 0, col0 = blockIdx.z * 64 + (FULL ? (wave >> 1) * 32 : wave * 16);
  const int col = col0 + r16;
  const bool col_ok = FULL || col < dv;
  const float* krow = a.vec + (size_t)row0 * a.width + a.k_col + (h / (a.H / a.G)) * dk + chan0 + (FULL ? r16 * CT : r16);
  const float* vrow = a.vec + (size_t)row0 * a.width + a.x_col + h * dv + (FULL ? col0 + r16 * VT : col_ok ? col : 0);
  f32x4_t kk[CT], v[VT];
  auto request = [&](int t0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // (tokens beyond the chunk have weight zero)
      const size_t at = (size_t)min(t0 + 4 * g + j, n - 1) * a.width;
      if constexpr (FULL) {
        const keys_t x = *reinterpret_cast<const keys_t*>(krow + at);
        const values_t y = *reinterpret_cast<const values_t*>(vrow + at);
#pragma unroll
        for (int t = 0; t < CT; ++t) kk[t][j] = x[t];
#pragma unroll
        for (int c = 0; c < VT; ++c) v[c][j] = y[c];
      } else {
        v[0][j] = col_ok ? vrow[at] : 0.f;
#pragma unroll
        for (int t = 0; t < NT; ++t) kk[t][j] = t * 16 + r16 < dk ? krow[at + t * 16] : 0.f;
      }
    }
  };
  request(0);

  // ---- c and dt of every token: two waves of 64 tokens each
  double c = 0.0;
  float dt = 0.f;
  if (tid < DC_CHUNK) {
    double l = 0.0;
    if (tid < n) {
      if (a.fixed) {
        dt = 1.f;
        l = log2((double)a.fixed[h]);
      } else {
        const size_t at = (size_t)(row0 + tid) * a.proj_stride + a.gate_col + h;
        const float raw = a.proj_bf16 ? (float)((const bf16_t*)a.proj)[at] : ((const float*)a.proj)[at];
        dt = softplus_f(raw + a.dt_bias[h]);
        l = (double)(-expf(a.A_log[h]) * dt) * 1.4426950408889634;
      }
      l = l < DC_LEAST_LOG2 ? DC_LEAST_LOG2 : l;
    }
    c = l;
#pragma unroll
    for (int o = 1; o < ZA_WAVE; o <<= 1) {
      const double v = __shfl_up(c, o, ZA_WAVE);
      if (lane >= o) c += v;
    }
    if (tid == 63) first_half = c;
  }
  __syncthreads();
  if (tid < DC_CHUNK) {
    if (wave == 1) c += first_half;
    if (tid == n - 1) whole = c;
  }
  __syncthreads();
  if (tid < DC_CHUNK) weight[tid] = tid < n ? (float)exp2(whole - c) * dt : 0.f;
  if (tid < n) {
    if (blockIdx.z == 0) {
      float* s = a.sums + ((size_t)(row0 + tid) * a.H + h) * 3;
      s[0] = (float)c;
      s[1] = (float)(c - (double)(float)c);
      s[2] = dt;
      if (tid == n - 1) a.total[(size_t)item * a.H + h] = (float)exp2(c);
    }
  }
  __syncthreads();

  f32x4_t S[VT][CT];
#pragma unroll
  for (int c = 0; c < VT; ++c)
#pragma unroll
    for (int t = 0; t < CT; ++t) S[c][t] = zero4();
  for (int t0 = 0; t0 < n; t0 += 16) {
    f32x4_t k0[CT], v0[VT];
    const f32x4_t w = *reinterpret_cast<const f32x4_t*>(&weight[t0 + 4 * g]);
#pragma unroll
    for (int c = 0; c < VT; ++c) v0[c] = v[c] * w;
#pragma unroll
    for (int t = 0; t < CT; ++t) k0[t] = kk[t];
    if (t0 + 16 < n) request(t0 + 16);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < VT; ++c)
#pragma unroll
        for (int t = 0; t < CT; ++t)
          S[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0[t][j], v0[c][j], S[c][t], 0, 0, 0);
  }
  if (!col_ok) return;
  if constexpr (FULL) {
    // row 4 g + i of all tiles: channels (4 g + i) * CT .. + CT - 1
#pragma unroll
    for (int c = 0; c < VT; ++c) {
      float* st = a.chunk_state + (((size_t)item * a.H + h) * dv + col0 + r16 * VT + c) * dk + chan0 + 4 * g * CT;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        keys_t x;
#pragma unroll
        for (int t = 0; t < CT; ++t) x[t] = S[c][t][i];
        *reinterpret_cast<keys_t*>(st + i * CT) = x;
      }
    }
    return;
  }
  float* st = a.chunk_state + (((size_t)item * a.H + h) * dv + col) * dk;
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int c4 = t * 16 + 4 * g;
    if (dk % 4 == 0) {
      if (c4 < dk) *reinterpret_cast<f32x4_t*>(st + c4) = S[0][t];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c4 + i < dk) st[c4 + i] = S[0][t][i];
    }
  }
}

// One thread a state element; the chunks of a request are neighbours in the list (a request without
// one is left alone).  Chunk states become the states before their chunks; the last one goes back
// to the request's slot.
__global__ void __launch_bounds__(256)
decay_prefix_kernel(float* __restrict__ chunk_state, float* __restrict__ state, long long slot_stride,
                    const int* __restrict__ slot_id, const int* __restrict__ item_seq, int n_items,
                    const float* __restrict__ total, int elems, int H, int per_head) {
  __shared__ int bounds[2];
  const int s = blockIdx.x, e = blockIdx.y * 256 + threadIdx.x;
  if (threadIdx.x == 0) { bounds[0] = n_items; bounds[1] = 0; }
  __syncthreads();
  for (int i = threadIdx.x; i < n_items; i += 256)
    if (item_seq[i] == s) {
      atomicMin(&bounds[0], i);
      atomicMax(&bounds[1], i + 1);
    }
  __syncthreads();
  const int first = bounds[0], last = bounds[1];
  if (e >= elems || first >= last) return;
  float* slot = state + (size_t)slot_id[s] * slot_stride + e;
  float S = *slot;
  for (int i0 = first; i0 < last; i0 += 8) {
    float local[8], a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = i0 + j < last;
      local[j] = in ? chunk_state[(size_t)(i0 + j) * elems + e] : 0.f;
      a[j] = in ? total[(size_t)(i0 + j) * H + e / per_head] : 1.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (i0 + j < last) chunk_state[(size_t)(i0 + j) * elems + e] = S;
      S = fmaf(a[j], S, local[j]);
    }
  }
  *slot = S;
}

// The scores of a chunk, once for all heads of a group (a head by itself works them out where it needs
// them): a workgroup a chunk, group and block of 16 tokens, its waves the blocks of keys in turn.
template <int NT, bool FULL>
__global__ void __launch_bounds__(256)
decay_chunk_scores_kernel(DecayArgs a) {
  const int item = blockIdx.x, grp = blockIdx.y, tile = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4;
  const int n = a.item_count[item], dk = a.dk;
  if (tile * 16 >= n) return;
  const float* rows = a.vec + (size_t)a.item_row0[item] * a.width;
  const bool aligned = dk % 4 == 0 && a.width % 4 == 0 && ((a.q_col | a.k_col) % 4) == 0 &&
                       (reinterpret_cast<uintptr_t>(a.vec) & 15) == 0;
  auto load = [&](int t0, int column, f32x4_t (&f)[NT]) {
    const float* p = rows + (size_t)min(t0 + r16, n - 1) * a.width + column + grp * dk;
#pragma unroll
    for (int t = 0; t < NT; ++t) f[t] = load4<FULL>(p + t * 16 + 4 * g, dk - (t * 16 + 4 * g), aligned);
  };
  f32x4_t fq[NT], fk[NT];
  load(tile * 16, a.q_col, fq);
  float* to = a.scores + (((size_t)item * a.G + grp) * DC_CHUNK + tile * 16 + r16) * DC_CHUNK + 4 * g;
  for (int J = wave; J <= tile; J += 4) {
    load(J * 16, a.k_col, fk);
    f32x4_t s = zero4(), u = zero4();
#pragma unroll
    for (int t = 0; t < NT; t += 2) {
      s = mfma4(fk[t], fq[t], s);
      if (t + 1 < NT) u = mfma4(fk[t + 1], fq[t + 1], u);
    }
    *reinterpret_cast<f32x4_t*>(to + J * 16) = s + u;
  }
}

// One workgroup a chunk, head and 64 columns; a wave takes two blocks of 16 tokens, one early and
// one late in the chunk, so that all waves meet the same number of earlier blocks.  The scores
// are taken turned round (keys along the rows), which is how the product with v reads them.
// SHARED: the scores come from decay_chunk_scores_kernel, and with them a key's dk elements stay away.
template <int NT, bool FULL, bool SHARED>
__global__ void __launch_bounds__(256, 2)
decay_chunk_out_kernel(DecayArgs a) {
  __shared__ float hi[DC_CHUNK], lo[DC_CHUNK], step[DC_CHUNK];
  // FULL: the 64 columns of the state before the chunk, a column's 16-byte pieces in the order piece ^ (column / 4 % 8)
  // (the eight columns read together fall into different banks)
  __shared__ __attribute__((aligned(16))) float Bs[FULL ? 64 * NT * 16 : 4];
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int row0 = a.item_row0[item], n = a.item_count[item];
  const int dk = a.dk, dv = a.dv, grp = h / (a.H / a.G);
  const float* B = a.chunk_state + ((size_t)item * a.H + h) * dv * dk;
  if constexpr (FULL) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int piece = (wave * NT + i) * 64 + lane, col = piece / (NT * 4);
      lds_request(B + (size_t)(blockIdx.z * 64 + col) * dk + ((piece % (NT * 4)) ^ (col >> 2 & 7)) * 4,
                  Bs + (wave * NT + i) * 256);
    }
  }
  const int blocks = (n + 15) / 16;
  const int tile[2] = {wave, 7 - wave};
  if (tid < DC_CHUNK) {
    const bool in = tid < n;
    const float* s = a.sums + ((size_t)(row0 + (in ? tid : 0)) * a.H + h) * 3;
    hi[tid] = in ? s[0] : 0.f;
    lo[tid] = in ? s[1] : 0.f;
    step[tid] = in ? s[2] : 0.f;
  }
  if constexpr (FULL) __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));      // (the state's pieces)
  __syncthreads();
  if (tile[0] >= blocks) return;
  const bool second = tile[1] < blocks;
  const int n0 = blockIdx.z * 64;
  // a lane's column of tile j: FULL: a lane's four are neighbours, read and written 16 bytes at a time
  auto col_of = [&](int j) { return n0 + (FULL ? 4 * r16 + j : j * 16 + r16); };
  const float* rows = a.vec + (size_t)row0 * a.width;
  const bool aligned = dk % 4 == 0 && a.width % 4 == 0 && ((a.q_col | a.k_col) % 4) == 0 &&
                       (reinterpret_cast<uintptr_t>(a.vec) & 15) == 0;

  f32x4_t fq[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float* q = rows + (size_t)min(tile[i] * 16 + r16, n - 1) * a.width + a.q_col + grp * dk;
#pragma unroll
    for (int t = 0; t < NT; ++t) fq[i][t] = load4<FULL>(q + t * 16 + 4 * g, dk - (t * 16 + 4 * g), aligned);
  }
  f32x4_t acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero4();

  // ---- what the state before the chunk gives
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    f32x4_t fb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = col_of(j);
      if constexpr (FULL)
        fb[j] = *reinterpret_cast<const f32x4_t*>(&Bs[(4 * r16 + j) * (NT * 16) + ((t * 4 + g) ^ (r16 & 7)) * 4]);
      else
        fb[j] = col < dv ? load4_below(B + (size_t)col * dk + t * 16 + 4 * g, dk - (t * 16 + 4 * g), dk % 4 == 0) : zero4();
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fq[i][t][e], fb[j][e], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = tile[i] * 16 + 4 * g + r;
      const float f = exp2_of(hi[tok], lo[tok]);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j][r] *= f;
    }

  // ---- what the chunk's own tokens give
  const int last = second ? tile[1] : tile[0];
  const float q_hi[2] = {hi[tile[0] * 16 + r16], hi[tile[1] * 16 + r16]};
  const float q_lo[2] = {lo[tile[0] * 16 + r16], lo[tile[1] * 16 + r16]};
  f32x4_t fk[SHARED ? 2 : NT], v[4];      // SHARED: the scores of both blocks of tokens
  [[maybe_unused]] const float* scored[2];
  if constexpr (SHARED)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      scored[i] = a.scores + (((size_t)item * a.G + grp) * DC_CHUNK + tile[i] * 16 + r16) * DC_CHUNK + 4 * g;
  auto request = [&](int J) {
    if constexpr (SHARED) {
#pragma unroll
      for (int i = 0; i < 2; ++i) fk[i] = *reinterpret_cast<const f32x4_t*>(scored[i] + J * 16);
    } else {
      const float* k = rows + (size_t)min(J * 16 + r16, n - 1) * a.width + a.k_col + grp * dk;
#pragma unroll
      for (int t = 0; t < NT; ++t) fk[t] = load4<FULL>(k + t * 16 + 4 * g, dk - (t * 16 + 4 * g), aligned);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // (no token sees one beyond the chunk)
      const float* x = rows + (size_t)min(J * 16 + 4 * g + r, n - 1) * a.width + a.x_col + h * dv;
      [[maybe_unused]] f32x4_t four;
      if constexpr (FULL) four = *reinterpret_cast<const f32x4_any_t*>(x + col_of(0));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (FULL) v[j][r] = four[j];
        else v[j][r] = col_of(j) < dv ? x[col_of(j)] : 0.f;
      }
    }
  };
  unsigned wild = 0;                 // of the blocks of own tokens and 16 columns: those with such numbers
  request(0);
  for (int J = 0; J <= last; ++J) {
    constexpr int KT = SHARED ? 2 : NT;
    f32x4_t k0[KT], v0[4];
#pragma unroll
    for (int t = 0; t < KT; ++t) k0[t] = fk[t];
#pragma unroll
    for (int j = 0; j < 4; ++j) v0[j] = v[j];
    if (J < last) request(J + 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (J > tile[i] || (i == 1 && !second)) continue;
      f32x4_t s = zero4();
      if constexpr (SHARED) {
        s = k0[i];
      } else {
        f32x4_t u = zero4();
#pragma unroll
        for (int t = 0; t < NT; t += 2) {
          s = mfma4(k0[t], fq[i][t], s);
          if (t + 1 < NT) u = mfma4(k0[t + 1], fq[i][t + 1], u);
        }
        s += u;
      }
      f32x4_t p;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = J * 16 + 4 * g + r;
        const float d = q_hi[i] - hi[key], lost = (q_hi[i] - d) - hi[key];
        p[r] = key <= tile[i] * 16 + r16 ? s[r] * (exp2_of(d, lost + (q_lo[i] - lo[key])) * step[key]) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4_t x = v0[j];
        if (J == tile[i] && any_wild(x)) {
          wild |= 1u << (i * 4 + j);
          x = without_wild(x);
        }
        acc[i][j] = mfma4(p, x, acc[i][j]);
      }
    }
  }
  if (wild)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (wild & (1u << (i * 4 + j))) {
          f32x4_t x;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int col = col_of(j);
            x[r] = FULL || col < dv
                       ? rows[(size_t)min(tile[i] * 16 + 4 * g + r, n - 1) * a.width + a.x_col + h * dv + col] : 0.f;
          }
          wild_from_its_row(x, acc[i][j], g);
        }
  const float D = a.D ? a.D[h] : 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (i == 1 && !second) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = tile[i] * 16 + 4 * g + r;
      if (tok >= n) continue;
      float* o = a.out + (size_t)(row0 + tok) * a.H * dv + h * dv;
      const float* x = rows + (size_t)tok * a.width + a.x_col + h * dv;
      if constexpr (FULL) {
        f32x4_t y = {acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
        if (a.D) {
          const f32x4_t four = *reinterpret_cast<const f32x4_any_t*>(x + col_of(0));
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = fmaf(D, four[j], y[j]);
        }
        *reinterpret_cast<f32x4_any_t*>(o + col_of(0)) = y;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int col = col_of(j);
          if (col < dv) o[col] = a.D ? fmaf(D, x[col], acc[i][j][r]) : acc[i][j][r];
        }
      }
    }
  }
}

// `items`: work items of at most DC_CHUNK rows, a request's side by side, of the requests that are
// taken (the others' rows of `out` and their states are left alone); scratch: `sums` n_tokens*H*3, `chunk_state` n_items*H*dv*dk, `total` n_items*H floats; `scores`
// n_items*G*128*128 floats where heads share their keys and queries, or null.
extern "C" int za_decay_chunked(const float* vec, int width, int q_col, int k_col, int x_col,
                                const void* proj, int dtype, int proj_stride, int gate_col,
                                const float* dt_bias, const float* A_log, const float* D,
                                const float* fixed, float* state, long long slot_stride,
                                const int* slot_id, const int* item_seq, const int* item_row0,
                                const int* item_count, int n_items, int n_seqs, float* sums,
                                float* chunk_state, float* total, float* scores, float* out, int n_tokens, int H,
                                int G, int dk, int dv, hipStream_t stream) {
  if (n_tokens == 0 || n_items == 0) return 0;
  if (n_tokens < 0 || n_seqs <= 0 || n_items < 0 || H <= 0 || G <= 0 || H % G || dk <= 0 || dv <= 0 ||
      !vec || !state || !slot_id || !item_seq || !item_row0 || !item_count || !sums || !chunk_state ||
      !total || !out || slot_stride < (long long)H * dk * dv)
    return ZA_ERR_ARG;
  if (!fixed && (!proj || !dt_bias || !A_log)) return ZA_ERR_ARG;
  if (dtype != 0 && dtype != 1) return ZA_ERR_UNSUPPORTED;
  const long long elems = (long long)H * dk * dv;
  if (dk > 128 || elems > 0x7fffffffLL || H > 65535) return ZA_ERR_UNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(scores) & 15) != 0) return ZA_ERR_ARG;
  const DecayArgs a{vec, width, q_col, k_col, x_col, proj, proj_stride, gate_col, dtype, dt_bias, A_log, D,
                    fixed, item_row0, item_count, sums, chunk_state, total, out, H, G, dk, dv, scores};
  dim3 grid(n_items, H, (dv + 63) / 64);
  const dim3 block(256);
  const bool full = dv % 64 == 0 && width % 4 == 0 && q_col % 4 == 0 && k_col % 4 == 0 &&
                    ((reinterpret_cast<uintptr_t>(vec) | reinterpret_cast<uintptr_t>(chunk_state)) & 15) == 0;
#define ZA_DECAY(KERNEL, ...)                                                                  \
  {                                                                                            \
    if (full && dk == 64) hipLaunchKernelGGL((KERNEL<4, true __VA_ARGS__>), grid, block, 0, stream, a);    \
    else if (full && dk == 128) hipLaunchKernelGGL((KERNEL<8, true __VA_ARGS__>), grid, block, 0, stream, a); \
    else if (dk <= 32) hipLaunchKernelGGL((KERNEL<2, false __VA_ARGS__>), grid, block, 0, stream, a);      \
    else if (dk <= 64) hipLaunchKernelGGL((KERNEL<4, false __VA_ARGS__>), grid, block, 0, stream, a);      \
    else hipLaunchKernelGGL((KERNEL<8, false __VA_ARGS__>), grid, block, 0, stream, a);                    \
    const int rc = za_launch_status();                                                         \
    if (rc != 0) return rc;                                                                    \
  }
#define ZA_COMMA ,
  ZA_DECAY(decay_chunk_state_kernel)
  hipLaunchKernelGGL(decay_prefix_kernel, dim3(n_seqs, (unsigned)((elems + 255) / 256)), dim3(256), 0, stream,
                     chunk_state, state, slot_stride, slot_id, item_seq, n_items, total, (int)elems, H, dk * dv);
  const int rc = za_launch_status();
  if (rc != 0) return rc;
  if (scores) {
    const dim3 by_heads = grid;
    grid = dim3(n_items, G, DC_CHUNK / 16);
    ZA_DECAY(decay_chunk_scores_kernel)
    grid = by_heads;
    ZA_DECAY(decay_chunk_out_kernel, ZA_COMMA true)
  } else {
    ZA_DECAY(decay_chunk_out_kernel, ZA_COMMA false)
  }
  return 0;
#undef ZA_COMMA
#undef ZA_DECAY
}

// ------------------------------------------------------------------- gated delta rule
//   S <- diag(g) S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// in chunks of 32 tokens.  With B the state before the chunk and P(j, i) the product of the decays
// of tokens j + 1 .. i (per key channel; P(i) from the chunk's start on, token i's included):
//   u_i = beta_i (v_i - B^T (P(i) k_i) - sum_(j < i) A_ij u_j),   A_ij = sum_c k_i k_j P(j, i)
//   o_i = B^T (P(i) q_i) + sum_(j <= i) Q_ij u_j,                 Q_ij = sum_c q_i k_j P(j, i)
//   S   = diag(P(n)) B + sum_j (P(j, n) k_j) u_j^T
// u is linear in B: u = U - W B, where U solves (1 + beta A) U = beta V and W the same with the
// rows P(i) k_i on the right, row after row, as the walk would meet them.
//   1. delta_chunk_prepare, all chunks and heads at once: U, W, Q, the scaled q, k and P(n)
//   2. delta_chunk_walk, one workgroup a request, head and 16 columns: chunk after chunk, the state
//      in registers
// Decays enter as products of themselves, never as quotients or logarithms: every factor is at
// most one when they are, and a decay of zero is nothing special.  Pairs of tokens within 16 take
// their product token by token; those of two neighbouring blocks of 16 as (product up to the
// first block's end) times (product from the second one's start on).
// 2,048 tokens, 16 heads of 128 x 128: 840 us walked token by token beside 38 us of preparation; 70 +
// 119 us here.  The walk over chunks is a chain of 1.9 us a chunk, 1.3 without any loads; of the
// rest some is its operands' way through the compute unit's cache (0.8 us more when every wave
// requested every operand).
#define DL_CHUNK 32

struct DeltaArgs {
  const float* conv;       // [T][conv_width]: q at q_col + g*dk, k at k_col + g*dk, v at x_col + h*dv
  int conv_width, q_col, k_col, x_col;
  const void* proj;        // [T][proj_stride] storage type: raw beta of head h at gate_col + h
  int proj_stride, gate_col;
  const void* decay;       // [T][decay_stride] storage type: the raw decay of head h and channel i at h*dk + i
  int decay_stride;
  const float* dt_bias;    // [H*dk]
  const float* A_log;      // [H]
  float* state;            // per slot [H][dv][dk]
  long long slot_stride;
  const int* slot_id;
  const int* item_seq;
  const int* item_row0;
  const int* item_count;
  int n_items;
  // a chunk's rows of one head lie side by side (a head's rows of consecutive tokens, a power of two
  // apart, meet in few of the cache's channels: 2,048 tokens walked in 186 us instead of 179)
  float* qp;               // [items][H][32][dk]: P(i) q_i
  float* W;                // [items][H][32][dk]
  float* U;                // [items][H][32][dv]
  float* Q;                // [items][H][32][32]: Q_ij, zeros for j > i
  float* kp;               // [items][H][dk][32]: P(j, n) k_j, zeros beyond the chunk's tokens
  float* grow;             // [items][H][dk]: P(n)
  float* out;              // [T][H*dv]
  int H, G, dk, dv;
};

// A barrier for what the workgroup shares in LDS only: the general one also waits for every load
// from memory under way, the next chunks' operands among them.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The sum over 16 neighbouring lanes, with the vector unit's own lane patterns.
template <int CTRL>
__device__ __forceinline__ float lane_add(float x) {
  const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false);
  return x + __builtin_bit_cast(float, moved);
}
__device__ __forceinline__ float sum16(float x) {
  return lane_add<0x140>(lane_add<0x141>(lane_add<0x4E>(lane_add<0xB1>(x))));
}

template <int DK, typename T>      // key channels, rounded up to 32, 64 or 128
__global__ void __launch_bounds__(256)
delta_chunk_prepare_kernel(DeltaArgs a) {
  constexpr int LD = DK + 4;
  // k and decays as they are; then k P(i) of the chunk for the solve; kx: k P(j, end of its block) of
  // the first block, k (product from its block's start on) of the second; qx the latter of q
  __shared__ __attribute__((aligned(16))) float ks[DL_CHUNK][LD], qs[DL_CHUNK][LD], gs[DL_CHUNK][LD];
  __shared__ __attribute__((aligned(16))) float A[DL_CHUNK][DL_CHUNK + 4];   // beta_i A_ij
  __shared__ float beta[DL_CHUNK];
  const int item = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g4 = lane >> 4;
  const int row0 = a.item_row0[item], n = a.item_count[item];
  const int dk = a.dk, dv = a.dv, grp = h / (a.H / a.G);
  const size_t at = (size_t)item * a.H + h;

  // ---- what the tokens bring (those beyond the chunk change nothing: no decay, nothing written
  // or read): unit q, times dk^(-1/2), and k; decays; write strengths
  const float neg_A = -expf(a.A_log[h]);
  {
    // (All requested before any is waited for, from rows and channels that are there: with a row
    // asked for once the one before had come, 2,048 tokens of 16 heads of 128 took 77.0 us instead
    // of 69.6, of 8 heads 40.2 instead of 36.7.)
    constexpr int PER = DL_CHUNK * DK / 256, ROWS = 256 / DK;
    const int c = tid % DK, ch = c < dk ? c : 0;
    float q[PER], k[PER], raw[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const size_t row = row0 + min(tid / DK + i * ROWS, n - 1);
      const float* x = a.conv + row * a.conv_width + grp * dk + ch;
      q[i] = x[a.q_col];
      k[i] = x[a.k_col];
      raw[i] = to_f32<T>(((const T*)a.decay)[row * a.decay_stride + h * dk + ch]);
    }
    const float bias = a.dt_bias[h * dk + ch];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int t = tid / DK + i * ROWS;
      const bool in = t < n && c < dk;
      qs[t][c] = in ? q[i] : 0.f;
      ks[t][c] = in ? k[i] : 0.f;
      gs[t][c] = in ? expf(neg_A * softplus_f(raw[i] + bias)) : 1.f;
    }
  }
  if (tid < DL_CHUNK) {
    const float raw = to_f32<T>(((const T*)a.proj)[(size_t)(row0 + min(tid, n - 1)) * a.proj_stride + a.gate_col + h]);
    beta[tid] = tid < n ? 1.0f / (1.0f + expf(-raw)) : 0.f;
  }
  __syncthreads();
  {
    // four lanes a vector
    const int t = (tid >> 2) & 31, sub = tid & 3;
    float* row = tid < 128 ? qs[t] : ks[t];
    float ss = 0.f;
#pragma unroll
    for (int c = sub * 4; c < DK; c += 16) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(row + c);
      ss += (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
    }
    ss = lane_add<0x4E>(lane_add<0xB1>(ss));
    float scale = 1.0f / sqrtf(ss + 1e-6f);
    if (tid < 128) scale *= 1.0f / sqrtf((float)dk);
#pragma unroll
    for (int c = sub * 4; c < DK; c += 16) {
      f32x4_t* x = reinterpret_cast<f32x4_t*>(row + c);
      *x *= scale;
    }
  }
  __syncthreads();

  // ---- pairs within a block of 16: a thread takes key j and DK / 16 channels, four at a time
  {
    const int j = tid >> 4, part = tid & 15;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float sk[16], sq[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) sk[i] = sq[i] = 0.f;
      for (int c = part * 4; c < DK; c += 64) {
        const f32x4_t kj = *reinterpret_cast<const f32x4_t*>(&ks[b * 16 + j][c]);
        f32x4_t p = zero4();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const f32x4_t ki = *reinterpret_cast<const f32x4_t*>(&ks[b * 16 + i][c]);
          const f32x4_t qi = *reinterpret_cast<const f32x4_t*>(&qs[b * 16 + i][c]);
          const f32x4_t gi = *reinterpret_cast<const f32x4_t*>(&gs[b * 16 + i][c]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            p[e] = i == j ? kj[e] : p[e] * gi[e];     // k_j P(j, i); zero before j
            sk[i] = fmaf(ki[e], p[e], sk[i]);
            sq[i] = fmaf(qi[e], p[e], sq[i]);
          }
          if (i % 2) __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float x = sum16(sk[i]), y = sum16(sq[i]);
        if (part == i) {
          A[b * 16 + i][b * 16 + j] = i > j ? beta[b * 16 + i] * x : 0.f;
          if (b * 16 + i < n)
            a.Q[(at * DL_CHUNK + b * 16 + i) * DL_CHUNK + b * 16 + j] = i >= j ? y : 0.f;
        }
      }
    }
  }
  __syncthreads();

  // ---- decays of every channel: a thread takes one channel's 16 tokens of one block
  const int c = tid % DK, b = tid / DK;
  const bool mine = tid < 2 * DK;
  float kbar[16];                       // P(i) k_i, for the solve
  if (mine) {
    float first = 1.f, own = 1.f;       // the product of the first block; of this one
#pragma unroll
    for (int i = 0; i < 16; ++i) first *= gs[i][c];
    float gk[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) gk[i] = gs[b * 16 + i][c];
    const float before = b == 0 ? 1.f : first;
    float last = 1.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) last *= gs[16 + i][c];
    float behind[16];                   // P(j, end of the block)
    own = 1.f;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      behind[i] = own;
      own *= gk[i];
    }
    const float after = b == 0 ? last : 1.f;
    float* kp = a.kp + (at * dk + (c < dk ? c : 0)) * DL_CHUNK + b * 16;
    float p = 1.f;
    float kx[16], qx[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = b * 16 + i;
      const float k = ks[t][c], q = qs[t][c];
      p *= gk[i];
      kbar[i] = k * (before * p);
      kx[i] = b == 0 ? k * behind[i] : k * p;
      qx[i] = q * p;
      if (c < dk && t < n) a.qp[(at * DL_CHUNK + t) * dk + c] = q * (before * p);
      behind[i] = k * (behind[i] * after);
    }
    if (c < dk) {
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<f32x4_t*>(kp + i) = f32x4_t{behind[i], behind[i + 1], behind[i + 2], behind[i + 3]};
      if (b == 1) a.grow[at * dk + c] = first * last;
    }
    // (nobody else reads this channel of the block's k and q here)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      ks[b * 16 + i][c] = kx[i];
      qs[b * 16 + i][c] = qx[i];
    }
  }
  __syncthreads();

  // ---- pairs of the second block's tokens with the first one's: two products of 16 x 16 x DK
  if (wave < 2) {
    const float(*left)[LD] = wave == 0 ? ks : qs;
    f32x4_t s = zero4();
#pragma unroll
    for (int t = 0; t < DK / 16; ++t)
      s = mfma4(*reinterpret_cast<const f32x4_t*>(&left[16 + r16][t * 16 + 4 * g4]),
                *reinterpret_cast<const f32x4_t*>(&ks[r16][t * 16 + 4 * g4]), s);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 + 4 * g4 + i;
      if (wave == 0) A[t][r16] = beta[t] * s[i];
      else if (t < n) a.Q[(at * DL_CHUNK + t) * DL_CHUNK + r16] = s[i];
    }
  } else if (wave == 2) {
    // (the first block's tokens see none of the second's)
    for (int i = lane; i < 256; i += 64)
      if (i / 16 < n) a.Q[(at * DL_CHUNK + i / 16) * DL_CHUNK + 16 + i % 16] = 0.f;
  }
  // the rows P(i) k_i take the decays' place
  __syncthreads();
  if (mine) {
#pragma unroll
    for (int i = 0; i < 16; ++i) gs[b * 16 + i][c] = kbar[i];
  }
  __syncthreads();

  // ---- the solve: a thread takes one column of V or of the rows P(i) k_i
  for (int col = tid; col < dv + dk; col += 256) {
    const bool of_v = col < dv;
    const float* v = a.conv + (size_t)row0 * a.conv_width + a.x_col + h * dv + (of_v ? col : 0);
    float y[DL_CHUNK];
#pragma unroll
    for (int i = 0; i < DL_CHUNK; ++i)
      y[i] = beta[i] * (!of_v ? gs[i][col - dv] : i < n ? v[(size_t)i * a.conv_width] : 0.f);
    int here = 0;
    asm volatile("" : "+v"(here));
#pragma unroll
    for (int i = 1; i < DL_CHUNK; ++i) {
      // (rows of A are read a few ahead: left alone the compiler reads all of them first, and has
      // no registers left)
      if (i > 3) asm volatile("" : "+v"(here), "+v"(y[i - 4]));
      f32x4_t s = zero4();
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const f32x4_t m = *reinterpret_cast<const f32x4_t*>(&A[i][j + here]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j + e < i) s[e] = fmaf(m[e], y[j + e], s[e]);
      }
      y[i] -= (s[0] + s[1]) + (s[2] + s[3]);
    }
    float* to = of_v ? a.U + at * DL_CHUNK * dv + col : a.W + at * DL_CHUNK * dk + col - dv;
    const int stride = of_v ? dv : dk;
#pragma unroll
    for (int i = 0; i < DL_CHUNK; ++i)
      if (i < n) to[i * stride] = y[i];
  }
}

// Chunk after chunk of one request, for one head and 16 columns.  Waves 0 to 3 keep the state, NT / 4
// (or one) tiles of 16 rows each, and its image in LDS, where all eight read it as an operand (a
// lane's four rows side by side, as the products leave them); a chunk is two products with the
// state, W B for u and (P q) B for o, each over two blocks of tokens and, in halves, over the
// rows, then the products with u.  Two barriers a chunk, the next three chunks' operands on their way.
// FULL: dk fills its tiles and dv its 16 columns.
template <int NT, bool FULL>
__global__ void __launch_bounds__(512)
delta_chunk_walk_kernel(DeltaArgs a) {
  constexpr int HT = NT / 2;                           // tiles of rows a half
  constexpr int OWN = NT >= 4 ? NT / 4 : 1;            // tiles of rows a wave keeps
  __shared__ f32x4_t Bs[NT][64], part[2][2][64], late[2][64];
  __shared__ int bounds[2];
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dk = a.dk, dv = a.dv;
  if (tid == 0) { bounds[0] = a.n_items; bounds[1] = 0; }
  __syncthreads();
  for (int i = tid; i < a.n_items; i += 512)
    if (a.item_seq[i] == s) {
      atomicMin(&bounds[0], i);
      atomicMax(&bounds[1], i + 1);
    }
  __syncthreads();
  const int first = __builtin_amdgcn_readfirstlane(bounds[0]), last = __builtin_amdgcn_readfirstlane(bounds[1]);
  if (first >= last) return;
  const int col = blockIdx.z * 16 + r16;
  const bool col_ok = col < dv, aligned = dk % 4 == 0;
  const bool keeper = wave < 4, has_rows = keeper && wave * OWN < NT;
  const int block = wave & 1, half = (wave >> 1) & 1;  // what this wave takes of a product with the state

  float* st = a.state + (size_t)a.slot_id[s] * a.slot_stride + ((size_t)h * dv + (col_ok ? col : 0)) * dk;
  const bool st_aligned = aligned && a.slot_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(a.state) & 15) == 0;
  f32x4_t S[OWN];
#pragma unroll
  for (int o = 0; o < OWN; ++o) S[o] = zero4();
  if (has_rows) {
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int c = (wave * OWN + o) * 16 + 4 * g;
      if (col_ok) S[o] = load4_below(st + c, dk - c, st_aligned);
      Bs[wave * OWN + o][lane] = S[o];
    }
  }

  const int begin = a.item_row0[first], end = a.item_row0[last - 1] + a.item_count[last - 1];
  // A chunk's operands are requested three chunks ahead: with one the way from memory outlasts a
  // chunk, and two leave 2,048 tokens of 16 heads of 128 at 126 us where three take 119 (8 heads 123
  // and 117; without any loads 84: the chain of products and barriers).  A use of some waits for a known number of later requests, so every chunk of a role makes
  // the same ones (beyond the last chunk for that one again).  A lane's places within a chunk; where
  // a chunk lies is the same for all lanes.  (The rows of a last chunk that has fewer than 32 are
  // there, but hold nothing: no use of them reaches a result.)
  const unsigned row_at = (unsigned)((block * 16 + r16) * dk + half * HT * 16 + 4 * g);
  auto request_left = [&](const float* of, int item, f32x4_t(&x)[HT]) {
    const float* rows = of + ((size_t)item * a.H + h) * DL_CHUNK * dk;
#pragma unroll
    for (int i = 0; i < HT; ++i)
      x[i] = load4<FULL>(rows + (row_at + i * 16), dk - ((half * HT + i) * 16 + 4 * g), aligned);
  };
  auto with_state = [&](const f32x4_t(&x)[HT], f32x4_t p) {
    f32x4_t q = zero4();
#pragma unroll
    for (int i = 0; i < HT; i += 2) {
      p = mfma4(x[i], Bs[half * HT + i][lane], p);
      if (i + 1 < HT) q = mfma4(x[i + 1], Bs[half * HT + i + 1][lane], q);
    }
    return p + q;
  };
  // u of one block of 16 tokens, zeros beyond the chunk
  auto u_of = [&](int item, int m) {
    const f32x4_t s = part[m][0][lane] + part[m][1][lane];
    const int n = end - begin - (item - first) * DL_CHUNK - m * 16 - 4 * g;
    f32x4_t u;
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = (FULL || col_ok) && i < n ? -s[i] : 0.f;
    return u;
  };

  if (keeper) {
    struct Operands {
      f32x4_t left[HT], own, kk[OWN][2], grow[OWN];
    };
    const int rows_of = min(wave * OWN, NT - OWN);
    const unsigned own_at = (unsigned)((block * 16 + 4 * g) * dv + (col_ok ? col : 0));
    const unsigned kk_at = (unsigned)((rows_of * 16 + r16) * DL_CHUNK + 4 * g);
    auto request = [&](int item, Operands& x) {
      const size_t at = (size_t)item * a.H + h;
      request_left(a.W, item, x.left);
#pragma unroll
      for (int i = 0; i < 4; ++i) x.own[i] = (a.U + (at * DL_CHUNK + i) * dv)[own_at];
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        const int c = (rows_of + o) * 16;
#pragma unroll
        for (int m = 0; m < 2; ++m)
          x.kk[o][m] = FULL || c + r16 < dk
                           ? *reinterpret_cast<const f32x4_t*>(a.kp + at * dk * DL_CHUNK +
                                                               (kk_at + o * 16 * DL_CHUNK + m * 16))
                           : zero4();
        x.grow[o] = load4<FULL>(a.grow + at * dk + c + 4 * g, dk - (c + 4 * g), aligned);
      }
    };
    auto chunk = [&](int item, Operands& x) {
      // W B - U, in halves (U last: it is the larger)
      const f32x4_t wb = with_state(x.left, zero4());
      part[block][half][lane] = half == 0 ? wb - x.own : wb;
      lds_barrier();
      const f32x4_t u[2] = {u_of(item, 0), u_of(item, 1)};
#pragma unroll
      for (int o = 0; o < OWN; ++o) S[o] = mfma4(x.kk[o][0], u[0], x.grow[o] * S[o]);
#pragma unroll
      for (int o = 0; o < OWN; ++o) S[o] = mfma4(x.kk[o][1], u[1], S[o]);
      if (has_rows) {
#pragma unroll
        for (int o = 0; o < OWN; ++o) Bs[wave * OWN + o][lane] = S[o];
      }
      request(min(item + 3, last - 1), x);
      lds_barrier();
    };
    Operands x, y, z;
    request(first, x);
    request(min(first + 1, last - 1), y);
    request(min(first + 2, last - 1), z);
    lds_barrier();
    int item = first;
    for (; item + 2 < last; item += 3) {
      chunk(item, x);
      chunk(item + 1, y);
      chunk(item + 2, z);
    }
    if (item < last) chunk(item, x);
    if (item + 1 < last) chunk(item + 1, y);
  } else {
    struct Operands {
      f32x4_t left[HT], q;
    };
    const unsigned q_at = (unsigned)((block * 16 + r16) * DL_CHUNK + half * 16 + 4 * g);
    auto request = [&](int item, Operands& x) {
      request_left(a.qp, item, x.left);
      x.q = *reinterpret_cast<const f32x4_t*>(a.Q + ((size_t)item * a.H + h) * DL_CHUNK * DL_CHUNK + q_at);
    };
    auto chunk = [&](int item, Operands& x) {
      f32x4_t p = with_state(x.left, zero4());
      lds_barrier();
      f32x4_t u = u_of(item, half);
      if (half >= block && any_wild(u)) {
        if (half == block) wild_from_its_row(u, p, g);      // (block 0 sees none of the second's)
        u = without_wild(u);
      }
      p = mfma4(x.q, u, p);
      if (half == 1) late[block][lane] = p;
      request(min(item + 3, last - 1), x);
      lds_barrier();
      if (half == 0 && col_ok) {
        p += late[block][lane];
        const int t = begin + (item - first) * DL_CHUNK + block * 16 + 4 * g;
        float* o = a.out + (size_t)t * a.H * dv + h * dv + col;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (t + i < end) o[(size_t)i * a.H * dv] = p[i];
      }
    };
    Operands x, y, z;
    request(first, x);
    request(min(first + 1, last - 1), y);
    request(min(first + 2, last - 1), z);
    lds_barrier();
    int item = first;
    for (; item + 2 < last; item += 3) {
      chunk(item, x);
      chunk(item + 1, y);
      chunk(item + 2, z);
    }
    if (item < last) chunk(item, x);
    if (item + 1 < last) chunk(item + 1, y);
  }
  if (!has_rows || !col_ok) return;
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int c = (wave * OWN + o) * 16 + 4 * g;
    if (st_aligned) {
      if (c < dk) *reinterpret_cast<f32x4_t*>(st + c) = S[o];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c + i < dk) st[c + i] = S[o][i];
    }
  }
}

// dtype: 0 = float32, 1 = bfloat16 (proj and decay).  `items`: work items of at most DL_CHUNK rows, a
// request's side by side and full but for its last, of the requests that are taken; scratch (floats, n_items times
// H of them each): qp, W and kp 32*dk, U 32*dv, Q 32*32, grow dk, all on 16 bytes.
extern "C" int za_delta_chunked(int dtype, const float* conv, int conv_width, int q_col, int k_col, int x_col,
                                const void* proj, int proj_stride, int gate_col, const void* decay,
                                int decay_stride, const float* dt_bias, const float* A_log, float* state,
                                long long slot_stride, const int* slot_id, const int* item_seq,
                                const int* item_row0, const int* item_count, int n_items, int n_seqs,
                                float* qp, float* W, float* U, float* Q, float* kp, float* grow, float* out,
                                int n_tokens, int H, int G, int dk, int dv, hipStream_t stream) {
  if (n_tokens == 0 || n_items == 0) return 0;
  if (n_tokens < 0 || n_seqs <= 0 || n_items < 0 || H <= 0 || G <= 0 || H % G || dk <= 0 || dv <= 0 || !conv ||
      !proj || !decay || !dt_bias || !A_log || !state || !slot_id || !item_seq || !item_row0 || !item_count ||
      !qp || !W || !U || !Q || !kp || !grow || !out || decay_stride < H * dk ||
      slot_stride < (long long)H * dk * dv)
    return ZA_ERR_ARG;
  if (dtype != 0 && dtype != 1) return ZA_ERR_UNSUPPORTED;
  if (dk > 128 || H > 65535 || (dv + 15) / 16 > 65535)
    return ZA_ERR_UNSUPPORTED;
  const DeltaArgs a{conv, conv_width, q_col, k_col, x_col, proj, proj_stride, gate_col, decay, decay_stride,
                    dt_bias, A_log, state, slot_stride, slot_id, item_seq, item_row0, item_count, n_items, qp,
                    W, U, Q, kp, grow, out, H, G, dk, dv};
  const dim3 chunks(n_items, H), walkers(n_seqs, H, (dv + 15) / 16);
  const bool full = dv % 16 == 0;
#define ZA_DELTA(DK)                                                                                             \
  {                                                                                                              \
    if (dtype == 0)                                                                                              \
      hipLaunchKernelGGL((delta_chunk_prepare_kernel<DK, float>), chunks, dim3(256), 0, stream, a);              \
    else                                                                                                         \
      hipLaunchKernelGGL((delta_chunk_prepare_kernel<DK, bf16_t>), chunks, dim3(256), 0, stream, a);             \
    const int rc = za_launch_status();                                                                           \
    if (rc != 0) return rc;                                                                                      \
    if (full && dk == DK)                                                                                        \
      hipLaunchKernelGGL((delta_chunk_walk_kernel<DK / 16, true>), walkers, dim3(512), 0, stream, a);            \
    else                                                                                                         \
      hipLaunchKernelGGL((delta_chunk_walk_kernel<DK / 16, false>), walkers, dim3(512), 0, stream, a);           \
    return za_launch_status();                                                                                   \
  }
  if (dk <= 32) ZA_DELTA(32)
  if (dk <= 64) ZA_DELTA(64)
  ZA_DELTA(128)
#undef ZA_DELTA
}
