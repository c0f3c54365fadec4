// Attention over one small latent vector a token ("latent attention"): what is cached for
// a token is a normed latent c [R] and, optionally, a rotated key part k_r [Dr] that all
// heads share; every head's keys and values are linear expansions of c,
//     k_h = Wuk_h c,   v_h = Wuv_h c.
// Neither is ever formed.  With q_h = [q_n | q_r] (unrotated | rotated),
//     q_h . [k_h | k_r] = (Wuk_h^T q_n) . c + q_r . k_r
//     sum_j p_j v_h,j   = Wuv_h (sum_j p_j c_j)
// so the attention runs with ONE key/value head whose key is the cached row [c | k_r]
// (W = R + Dr elements) and whose value is the row's first R elements, with queries
// [Wuk_h^T q_n | q_r] and results that the head's Wuv expands afterwards.  The cache holds
// one plane of W elements a token, rows of a page one after the other.
//
// Kernels:
//   latent_prepare     a token's opening projection -> the normed query latent, and the row
//                      [rmsnorm(c) | rotate(k_r)] into the token's place in the cache
//   rotate_part        the rotated part of every head's query into the folded query
//   head_linear        out[t][h] = x[t][h] @ W[h]^T for every head at once (the two
//                      foldings above), optionally times sigmoid(gate) a head or an element
//   latent_attention   the attention itself: causal, streaming softmax in 32-bit with a sink
//                      a head, any mix of prompt portions and single tokens in one launch,
//                      contexts optionally cut into ranges (latent_combine merges them)
//   latent_prefill_mfma     the same on the matrix cores for prompt portions and mixed steps:
//                      latents of 128, 256 or 512 with up to 64 rotated elements
//   latent_attention_mfma   the same for other widths (bfloat16, 16-byte pieces): four waves of
//                      16 rows each
//   latent_decode_mfma      steps that only decode: four waves share 16 rows
// Rotation: adjacent pairs (2i, 2i + 1) or halves (i, i + dims/2) of the first `rot_dims`
// elements, angle = position * inv_freq[i] in 32-bit, cosine and sine times `magnitude`.
#include <math.h>

#include <type_traits>

#include "common.h"
#include "tiles_bf16.h"

// ------------------------------------------------------------------ latent_prepare
// down: [T][ld], columns [q_col, q_col + Rq) the query latent, [c_col, c_col + R) the
// latent, then Dr elements of the rotated key part.  cq: [T][Rq].  plane: the cache,
// token t's row at plane + (slots[t] / page_size) * page_stride + (slots[t] % page_size) * W.
template <typename T>
__global__ void __launch_bounds__(256)
latent_prepare_kernel(const T* __restrict__ down, int ld, int q_col, int Rq, int c_col, int R,
                      int Dr, const float* __restrict__ q_norm_w, const float* __restrict__ c_norm_w,
                      float eps, const int* __restrict__ positions, const int* __restrict__ slots,
                      const float* __restrict__ inv_freq, int rot_dims, int adjacent,
                      float magnitude, T* __restrict__ cq, T* __restrict__ plane, int page_size,
                      long long page_stride) {
  __shared__ float scratch[16];
  const size_t t = blockIdx.x;
  const T* row = down + t * ld;
  const int tid = threadIdx.x, bd = blockDim.x;
  if (cq) {
    float ss = 0.f;
    for (int i = tid; i < Rq; i += bd) {
      const float v = to_f32<T>(row[q_col + i]);
      ss += v * v;
    }
    ss = block_sum(ss, scratch);
    const float f = 1.0f / sqrtf(ss / (float)Rq + eps);
    for (int i = tid; i < Rq; i += bd)
      cq[t * Rq + i] = from_f32<T>(to_f32<T>(row[q_col + i]) * f * q_norm_w[i]);
  }
  if (!plane) return;
  const int slot = slots[t];
  if (slot < 0) return;
  T* dst = plane + (size_t)(slot / page_size) * page_stride + (size_t)(slot % page_size) * (R + Dr);
  float ss = 0.f;
  for (int i = tid; i < R; i += bd) {
    const float v = to_f32<T>(row[c_col + i]);
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float f = 1.0f / sqrtf(ss / (float)R + eps);
  for (int i = tid; i < R; i += bd)
    dst[i] = from_f32<T>(to_f32<T>(row[c_col + i]) * f * c_norm_w[i]);
  const T* kr = row + c_col + R;
  const int half = rot_dims / 2;
  const float pos = (float)positions[t];
  for (int i = tid; i < half; i += bd) {
    const int a = adjacent ? 2 * i : i, b = adjacent ? 2 * i + 1 : i + half;
    float sn, cs;
    sincosf(pos * inv_freq[i], &sn, &cs);
    sn *= magnitude;
    cs *= magnitude;
    const float u = to_f32<T>(kr[a]), v = to_f32<T>(kr[b]);
    dst[R + a] = from_f32<T>(u * cs - v * sn);
    dst[R + b] = from_f32<T>(v * cs + u * sn);
  }
  for (int i = rot_dims + tid; i < Dr; i += bd) dst[R + i] = kr[i];
}

// The same for a query latent of at most 256 * LP_Q elements, a latent of at most 256 * LP_C and a
// rotated part of at most 256: everything a token needs is requested at once, the two sums of
// squares meet at once, and nothing is read a second time.  (One way to memory bounds it: eight
// tokens with latents of 1,536 and 512 7.4 us in a step, 9.3 with the kernel above.)
#define LP_Q 8
#define LP_C 2
template <typename T>
__global__ void __launch_bounds__(256)
latent_prepare_regs_kernel(const T* __restrict__ down, int ld, int q_col, int Rq, int c_col, int R,
                           int Dr, const float* __restrict__ q_norm_w,
                           const float* __restrict__ c_norm_w, float eps,
                           const int* __restrict__ positions, const int* __restrict__ slots,
                           const float* __restrict__ inv_freq, int rot_dims, int adjacent,
                           float magnitude, T* __restrict__ cq, T* __restrict__ plane, int page_size,
                           long long page_stride) {
  __shared__ float part[4][2];
  const size_t t = blockIdx.x;
  const T* row = down + t * ld;
  const int tid = threadIdx.x;
  float qv[LP_Q], qw[LP_Q], cv[LP_C], cw[LP_C], u = 0.f, v = 0.f, freq = 0.f, pos = 0.f;
  int slot = -1;
  const int half = rot_dims / 2;
  const int a = adjacent ? 2 * tid : tid, b = adjacent ? 2 * tid + 1 : tid + half;
#pragma unroll
  for (int k = 0; k < LP_Q; ++k) {
    const int i = min(tid + k * 256, Rq - 1);
    qv[k] = cq ? to_f32<T>(row[q_col + i]) : 0.f;
    qw[k] = cq ? q_norm_w[i] : 0.f;
  }
  if (plane) {
    slot = slots[t];
#pragma unroll
    for (int k = 0; k < LP_C; ++k) {
      const int i = min(tid + k * 256, R - 1);
      cv[k] = to_f32<T>(row[c_col + i]);
      cw[k] = c_norm_w[i];
    }
    const T* kr = row + c_col + R;
    if (tid < half) {
      u = to_f32<T>(kr[a]);
      v = to_f32<T>(kr[b]);
      freq = inv_freq[tid];
      pos = (float)positions[t];
    } else if (rot_dims + tid - half < Dr) {
      u = to_f32<T>(kr[rot_dims + tid - half]);
    }
  }
  float sq = 0.f, sc = 0.f;
#pragma unroll
  for (int k = 0; k < LP_Q; ++k) sq += tid + k * 256 < Rq ? qv[k] * qv[k] : 0.f;
  if (plane)
#pragma unroll
    for (int k = 0; k < LP_C; ++k) sc += tid + k * 256 < R ? cv[k] * cv[k] : 0.f;
  sq = wave_sum(sq);
  sc = wave_sum(sc);
  if ((tid & 63) == 0) {
    part[tid >> 6][0] = sq;
    part[tid >> 6][1] = sc;
  }
  __syncthreads();
  sq = part[0][0] + part[1][0] + part[2][0] + part[3][0];
  sc = part[0][1] + part[1][1] + part[2][1] + part[3][1];
  if (cq) {
    const float f = 1.0f / sqrtf(sq / (float)Rq + eps);
#pragma unroll
    for (int k = 0; k < LP_Q; ++k) {
      const int i = tid + k * 256;
      if (i < Rq) cq[t * Rq + i] = from_f32<T>(qv[k] * f * qw[k]);
    }
  }
  if (slot < 0) return;
  T* dst = plane + (size_t)(slot / page_size) * page_stride + (size_t)(slot % page_size) * (R + Dr);
  const float f = 1.0f / sqrtf(sc / (float)R + eps);
#pragma unroll
  for (int k = 0; k < LP_C; ++k) {
    const int i = tid + k * 256;
    if (i < R) dst[i] = from_f32<T>(cv[k] * f * cw[k]);
  }
  if (tid < half) {
    float sn, cs;
    sincosf(pos * freq, &sn, &cs);
    sn *= magnitude;
    cs *= magnitude;
    dst[R + a] = from_f32<T>(u * cs - v * sn);
    dst[R + b] = from_f32<T>(v * cs + u * sn);
  } else if (rot_dims + tid - half < Dr) {
    dst[R + rot_dims + tid - half] = from_f32<T>(u);
  }
}

extern "C" int za_latent_prepare(const void* down, int dtype, int ld, int q_col, int q_rank,
                                 int c_col, int kv_rank, int rot_dim, const float* q_norm_w,
                                 const float* c_norm_w, float eps, const int* positions,
                                 const int* slots, const float* inv_freq, int rot_dims,
                                 int adjacent, float magnitude, void* cq, void* plane, int page_size,
                                 long long page_stride, int n_tokens, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || !down || ld <= 0 || kv_rank <= 0 || rot_dim < 0 || rot_dims < 0 ||
      rot_dims > rot_dim || rot_dims % 2 != 0 || c_col < 0 ||
      (plane && c_col + kv_rank + rot_dim > ld) ||
      (cq && (q_rank <= 0 || q_col < 0 || q_col + q_rank > ld || !q_norm_w)) ||
      (plane && (!slots || !c_norm_w || page_size <= 0 || page_stride < (long long)page_size * (kv_rank + rot_dim))) ||
      (plane && rot_dims > 0 && (!inv_freq || !positions)))
    return ZA_ERR_ARG;
  dim3 grid(n_tokens), block(256);
  // (a thread has one pair of the rotated part, or one element behind the rotated ones)
  const bool regs = (!cq || q_rank <= 256 * LP_Q) &&
                    (!plane || (kv_rank <= 256 * LP_C && rot_dim - rot_dims / 2 <= 256));
#define ZA_LP(T)                                                                                     \
  do {                                                                                               \
    if (regs)                                                                                        \
      hipLaunchKernelGGL((latent_prepare_regs_kernel<T>), grid, block, 0, stream, (const T*)down, ld, q_col, \
                         q_rank, c_col, kv_rank, rot_dim, q_norm_w, c_norm_w, eps, positions, slots, \
                         inv_freq, rot_dims, adjacent, magnitude, (T*)cq, (T*)plane, page_size,      \
                         page_stride);                                                               \
    else                                                                                             \
      hipLaunchKernelGGL((latent_prepare_kernel<T>), grid, block, 0, stream, (const T*)down, ld, q_col,      \
                         q_rank, c_col, kv_rank, rot_dim, q_norm_w, c_norm_w, eps, positions, slots, \
                         inv_freq, rot_dims, adjacent, magnitude, (T*)cq, (T*)plane, page_size,      \
                         page_stride);                                                               \
  } while (0)
  if (dtype == 0) ZA_LP(float);
  else if (dtype == 1) ZA_LP(bf16_t);
#undef ZA_LP
  else
    return ZA_ERR_UNSUPPORTED;
  return za_launch_status();
}

// --------------------------------------------------------------------- rotate_part
// dst[t][h][dst_col + i] = rotation of src[t][h][src_col + i], i < Dr (elements beyond
// rot_dims are copied).  One thread a pair.
template <typename T>
__device__ __forceinline__ void rotate_pair(const T* s, T* d, int i, int position, const float* __restrict__ inv_freq,
                                            int rot_dims, int adjacent, float magnitude) {
  const int half = rot_dims / 2;
  if (i < half) {
    const int a = adjacent ? 2 * i : i, b = adjacent ? 2 * i + 1 : i + half;
    float sn, cs;
    sincosf((float)position * inv_freq[i], &sn, &cs);
    sn *= magnitude;
    cs *= magnitude;
    const float u = to_f32<T>(s[a]), v = to_f32<T>(s[b]);
    d[a] = from_f32<T>(u * cs - v * sn);
    d[b] = from_f32<T>(v * cs + u * sn);
  } else {
    const int e = rot_dims + (i - half);
    d[e] = s[e];
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
rotate_part_kernel(const T* __restrict__ src, int src_ld, int src_col, T* __restrict__ dst,
                   int dst_ld, int dst_col, int H, int Dr, const int* __restrict__ positions,
                   const float* __restrict__ inv_freq, int rot_dims, int adjacent, float magnitude,
                   size_t total) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int per = Dr - rot_dims / 2;         // pairs, then the elements that pass unchanged
  const size_t th = idx / per;               // token * H + head
  rotate_pair<T>(src + th * src_ld + src_col, dst + th * dst_ld + dst_col, (int)(idx % per), positions[th / H], inv_freq,
                 rot_dims, adjacent, magnitude);
}

extern "C" int za_rotate_part(const void* src, int dtype, int src_ld, int src_col, void* dst,
                              int dst_ld, int dst_col, int n_tokens, int heads, int rot_dim,
                              const int* positions, const float* inv_freq, int rot_dims,
                              int adjacent, float magnitude, hipStream_t stream) {
  if (n_tokens == 0 || rot_dim == 0) return 0;
  if (n_tokens < 0 || heads <= 0 || rot_dim < 0 || rot_dims < 0 || rot_dims > rot_dim ||
      rot_dims % 2 != 0 || !src || !dst || src_col < 0 || dst_col < 0 ||
      src_col + rot_dim > src_ld || dst_col + rot_dim > dst_ld ||
      (rot_dims > 0 && (!positions || !inv_freq)))
    return ZA_ERR_ARG;
  const size_t total = (size_t)n_tokens * heads * (rot_dim - rot_dims / 2);
  dim3 grid((unsigned)((total + 255) / 256)), block(256);
  if (dtype == 0)
    hipLaunchKernelGGL((rotate_part_kernel<float>), grid, block, 0, stream, (const float*)src,
                       src_ld, src_col, (float*)dst, dst_ld, dst_col, heads, rot_dim, positions,
                       inv_freq, rot_dims, adjacent, magnitude, total);
  else if (dtype == 1)
    hipLaunchKernelGGL((rotate_part_kernel<bf16_t>), grid, block, 0, stream, (const bf16_t*)src,
                       src_ld, src_col, (bf16_t*)dst, dst_ld, dst_col, heads, rot_dim, positions,
                       inv_freq, rot_dims, adjacent, magnitude, total);
  else
    return ZA_ERR_UNSUPPORTED;
  return za_launch_status();
}

// --------------------------------------------------------------------- head_linear
// out[t][h][o_col + n] = (sum_k x[t][h][x_col + k] * W[h][n][k]) * gate(t, h, n)
//   x:   [T][H][x_ld]      W: [H][N][K]      out: [T][H][o_ld]
//   gate_mode 0: none; 1: sigmoid(gate[t][gate_col + h]); 2: sigmoid(gate[t][gate_col + h*N + n])
// Every output element is a sum over k in an order fixed by K alone.
struct HeadLinearArgs {
  const void* x;
  const void* W;
  void* out;
  const void* gate;
  int T, H, N, K;
  int x_ld, x_col, o_ld, o_col;
  int gate_ld, gate_col, gate_mode;
  // Dr > 0: a further workgroup a head rotates x's columns rot_src .. into out's columns rot_dst .. (rotate_pair)
  int Dr, rot_src, rot_dst, rot_dims, adjacent;
  float magnitude;
  const int* positions;
  const float* inv_freq;
};

template <typename TG>
__device__ __forceinline__ float head_gate_of(const HeadLinearArgs& a, int t, int h, int n) {
  if (a.gate_mode == 0) return 1.0f;
  const TG* g = (const TG*)a.gate + (size_t)t * a.gate_ld + a.gate_col;
  const float z = to_f32<TG>(a.gate_mode == 1 ? g[h] : g[(size_t)h * a.N + n]);
  return 1.0f / (1.0f + expf(-z));
}

// A decode batch (at most 16 rows), bfloat16 on the matrix cores, operands straight from memory into
// the fragments (layout: tiles_bf16.h), 128 elements of K under way at once a wave.  SPLIT: a
// workgroup has 16 columns of one head, its four waves a quarter of K each, which meet in LDS;
// otherwise 64 columns, 16 a wave.  What bounds it is the way to memory and back, once with K up to
// 512: 8 rows of 16 heads, [128 x 512] with a gate an element 2.9 us (64 columns a workgroup, a
// wave the whole of K in steps of 64: 5.8); [512 x 128] 3.1 (SPLIT 3.6: so from K = 256 on).
#define HL_SPLIT_MIN_K 256
template <typename TO, bool SPLIT>
__global__ void __launch_bounds__(256)
head_linear_rows16_kernel(HeadLinearArgs a) {
  __shared__ __attribute__((aligned(16))) float part[SPLIT ? 4 : 1][16][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = blockIdx.z, n0 = SPLIT ? blockIdx.y * 16 : blockIdx.y * 64 + wave * 16;
  const int r16 = lane & 15, kq = lane >> 4;
  const int K = a.K, N = a.N;
  if constexpr (!SPLIT && std::is_same<TO, bf16_t>::value)
    if (a.Dr > 0 && blockIdx.y == gridDim.y - 1) {
      const int per = a.Dr - a.rot_dims / 2;
      for (int idx = tid; idx < a.T * per; idx += 256) {
        const int t = idx / per;
        const size_t th = (size_t)t * a.H + h;
        rotate_pair<bf16_t>((const bf16_t*)a.x + th * a.x_ld + a.rot_src, (bf16_t*)a.out + th * a.o_ld + a.rot_dst,
                            idx - t * per, a.positions[t], a.inv_freq, a.rot_dims, a.adjacent, a.magnitude);
      }
      return;
    }
  const int range = SPLIT ? (K + 127) / 128 * 32 : K, k_lo = SPLIT ? wave * range : 0;
  const int k_end = min(K, k_lo + range);
  const bf16_t* arow = (const bf16_t*)a.x + ((size_t)min(r16, a.T - 1) * a.H + h) * a.x_ld + a.x_col;
  const bf16_t* wrow = (const bf16_t*)a.W + ((size_t)h * N + min(n0 + r16, N - 1)) * K;
  // SPLIT: the element that this thread stores; its gate on its way with the operands
  const int st = tid >> 4, sn = n0 + (tid & 15);
  const bool mine = SPLIT && st < a.T && sn < N;
  const float gate = mine ? head_gate_of<bf16_t>(a, st, h, sn) : 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
  constexpr int U = 4;
  for (int k0 = k_lo; k0 < k_end; k0 += 32 * U) {
    bf16x8_t fa[U], fw[U];
#pragma unroll
    for (int s = 0; s < U; ++s) {          // K is a multiple of 8: a piece is inside or outside
      const int k = min(k0 + s * 32 + kq * 8, K - 8);
      fa[s] = *reinterpret_cast<const bf16x8_t*>(arow + k);
      fw[s] = *reinterpret_cast<const bf16x8_t*>(wrow + k);
    }
#pragma unroll
    for (int s = 0; s < U; ++s) {
      if (k0 + s * 32 + kq * 8 >= k_end) fa[s] = fw[s] = zero;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[s], fw[s], acc, 0, 0, 0);
    }
  }
  TO* out = (TO*)a.out + a.o_col;
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = 0; i < 4; ++i) part[wave][kq * 4 + i][r16] = acc[i];
    __syncthreads();
    if (!mine) return;
    const int c = tid & 15;
    const float v = (part[0][st][c] + part[1][st][c]) + (part[2][st][c] + part[3][st][c]);
    out[((size_t)st * a.H + h) * a.o_ld + sn] = from_f32<TO>(v * gate);
  } else {
    const int n = n0 + r16;
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = kq * 4 + i;
      if (t < a.T)
        out[((size_t)t * a.H + h) * a.o_ld + n] = from_f32<TO>(acc[i] * head_gate_of<bf16_t>(a, t, h, n));
    }
  }
}

// The same for more rows than a decode batch has, in tiles of BM tokens x 128 columns of one head
// through LDS (tiles_bf16.h); a lane has four consecutive columns of a token's row.  With many
// tokens the result's way to memory bounds it ([1777, 16 heads, 512], rows of 576, from 128: 17 us
// against 37 of fragments straight from memory; [1777, 16, 128] with gates from 512: 15 against
// 44), with few the steps of K, one after the other (64 tokens: 4.0 against 5.3, 9.0 against 14.7).
// Tiles of 128 tokens: 21 and 27 us.
#define HL_BN 128
template <int BM, int NS, typename TO>
__global__ void __launch_bounds__(256, 2)
head_linear_tiled_kernel(HeadLinearArgs a) {
  using Tiles = TilesBf16<BM, HL_BN, NS>;
  __shared__ __attribute__((aligned(16))) bf16_t As[NS][BM * GG_BK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[NS][HL_BN * GG_BK];
  const int h = blockIdx.z, t0 = blockIdx.x * BM, n0 = blockIdx.y * HL_BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K, N = a.N;
  const int lrow = wave * 8 + (lane >> 3), piece = (lane & 7) ^ (lane >> 3);
  const bf16_t* arow[Tiles::LA];
  const bf16_t* wrow[Tiles::LW];
#pragma unroll
  for (int i = 0; i < Tiles::LA; ++i)
    arow[i] = (const bf16_t*)a.x + ((size_t)min(t0 + lrow + 32 * i, a.T - 1) * a.H + h) * a.x_ld + a.x_col + piece * 8;
#pragma unroll
  for (int i = 0; i < Tiles::LW; ++i)
    wrow[i] = (const bf16_t*)a.W + ((size_t)h * N + min(n0 + lrow + 32 * i, N - 1)) * K + piece * 8;
  const int wm = (wave % Tiles::WM) * (BM / Tiles::WM), wn = (wave / Tiles::WM) * (HL_BN / Tiles::WN);
  const int r16 = lane & 15, kq = lane >> 4;
  // a gate an element, four at a time and all at once, before the products
  const bool gates = a.gate_mode == 2 && ((a.gate_ld | a.gate_col | N) & 3) == 0 &&
                     (reinterpret_cast<uintptr_t>(a.gate) & 7) == 0;
  bf16x4_t gate[Tiles::TM][Tiles::TN];
  if (gates)
#pragma unroll
    for (int i = 0; i < Tiles::TM; ++i)
#pragma unroll
      for (int j = 0; j < Tiles::TN; ++j)
        gate[i][j] = *reinterpret_cast<const bf16x4_t*>(
            (const bf16_t*)a.gate + (size_t)min(t0 + wm + i * 16 + r16, a.T - 1) * a.gate_ld + a.gate_col +
            (size_t)h * N + min(n0 + wn + j * 16 + kq * 4, N - 4));
  f32x4_t acc[Tiles::TM][Tiles::TN];
  Tiles::run(As, Ws, wave, lane, K, arow, wrow, acc);
  TO* out = (TO*)a.out;
  const bool wide = ((a.o_ld | a.o_col | N) & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & (4 * sizeof(TO) - 1)) == 0;
#pragma unroll
  for (int i = 0; i < Tiles::TM; ++i) {
    const int t = t0 + wm + i * 16 + r16;
    if (t >= a.T) continue;
    TO* to = out + ((size_t)t * a.H + h) * a.o_ld + a.o_col;
#pragma unroll
    for (int j = 0; j < Tiles::TN; ++j) {
      const int n = n0 + wn + j * 16 + kq * 4;
      if (n >= N) continue;
      f32x4_t v = acc[i][j];
      if (a.gate_mode == 2 && gates) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= 1.0f / (1.0f + expf(-(float)gate[i][j][r]));
      } else if (a.gate_mode) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= head_gate_of<bf16_t>(a, t, h, min(n + r, N - 1));
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

// 32-bit weights (x of either type): 64 x 64 tiles through LDS, plain FMA.
template <typename TA, typename TO>
__global__ void __launch_bounds__(256)
head_linear_f32_kernel(HeadLinearArgs a) {
  __shared__ float As[16][64 + 4];
  __shared__ float Ws[16][64 + 4];
  const int h = blockIdx.z;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const int n0 = blockIdx.y * 64, m0 = blockIdx.x * 64;
  const int K = a.K, N = a.N;
  const float* W = (const float*)a.W + (size_t)h * N * K;
  const int lrow = tid / 4, lk = (tid % 4) * 4;
  const bool a_ok = m0 + lrow < a.T;
  const TA* arow = (const TA*)a.x + ((size_t)(a_ok ? m0 + lrow : 0) * a.H + h) * a.x_ld + a.x_col;
  const bool w_ok = n0 + lrow < N;
  const float* wrow = W + (size_t)(w_ok ? n0 + lrow : 0) * K;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      As[lk + j][lrow] = (a_ok && k < K) ? to_f32<TA>(arow[k]) : 0.f;
      Ws[lk + j][lrow] = (w_ok && k < K) ? wrow[k] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
  TO* out = (TO*)a.out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = m0 + ty * 4 + i;
    if (r >= a.T) continue;
    TO* orow = out + ((size_t)r * a.H + h) * a.o_ld + a.o_col;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) orow[n] = from_f32<TO>(acc[i][j] * head_gate_of<TA>(a, r, h, n));
    }
  }
}

// dtype codes: 0 = float32, 1 = bfloat16.  The gate has x's type.
extern "C" int za_head_linear(const void* x, int x_dtype, int x_ld, int x_col, const void* W,
                              int w_dtype, void* out, int out_dtype, int o_ld, int o_col,
                              int n_tokens, int heads, int N, int K, const void* gate, int gate_ld,
                              int gate_col, int gate_mode, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || heads <= 0 || heads > 65535 || N <= 0 || K <= 0 || !x || !W || !out ||
      x_col < 0 || o_col < 0 || x_col + K > x_ld || o_col + N > o_ld || gate_mode < 0 ||
      gate_mode > 2 || (gate_mode && (!gate || gate_col < 0)) ||
      (gate_mode == 1 && gate_col + heads > gate_ld) ||
      (gate_mode == 2 && (long long)gate_col + (long long)heads * N > gate_ld))
    return ZA_ERR_ARG;
  HeadLinearArgs a{x, W, out, gate, n_tokens, heads, N, K, x_ld, x_col, o_ld, o_col,
                   gate_ld, gate_col, gate_mode, 0, 0, 0, 0, 0, 0.f, nullptr, nullptr};
  if (w_dtype == 1) {
    if (x_dtype != 1 || K % 8 != 0 || x_ld % 8 != 0 || x_col % 8 != 0 || ((uintptr_t)x | (uintptr_t)W) % 16 != 0)
      return ZA_ERR_UNSUPPORTED;
    if (out_dtype != 0 && out_dtype != 1) return ZA_ERR_UNSUPPORTED;
    if (n_tokens <= 16) {
      const bool split = K >= HL_SPLIT_MIN_K;
      dim3 grid(1, (unsigned)(split ? (N + 15) / 16 : (N + 63) / 64), heads);
#define ZA_HL(TO, SPLIT) hipLaunchKernelGGL((head_linear_rows16_kernel<TO, SPLIT>), grid, dim3(256), 0, stream, a)
      if (out_dtype == 0) { if (split) ZA_HL(float, true); else ZA_HL(float, false); }
      else { if (split) ZA_HL(bf16_t, true); else ZA_HL(bf16_t, false); }
#undef ZA_HL
      return za_launch_status();
    }
    dim3 grid((unsigned)((n_tokens + 63) / 64), (unsigned)((N + HL_BN - 1) / HL_BN), heads);
    if (out_dtype == 0)
      hipLaunchKernelGGL((head_linear_tiled_kernel<64, 2, float>), grid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((head_linear_tiled_kernel<64, 2, bf16_t>), grid, dim3(256), 0, stream, a);
    return za_launch_status();
  }
  if (w_dtype != 0) return ZA_ERR_UNSUPPORTED;
  dim3 grid((unsigned)((n_tokens + 63) / 64), (unsigned)((N + 63) / 64), heads);
#define ZA_HF(TA, TO) \
  hipLaunchKernelGGL((head_linear_f32_kernel<TA, TO>), grid, dim3(256), 0, stream, a)
  if (x_dtype == 0 && out_dtype == 0) ZA_HF(float, float);
  else if (x_dtype == 1 && out_dtype == 0) ZA_HF(bf16_t, float);
  else if (x_dtype == 1 && out_dtype == 1) ZA_HF(bf16_t, bf16_t);
  else if (x_dtype == 0 && out_dtype == 1) ZA_HF(float, bf16_t);
  else return ZA_ERR_UNSUPPORTED;
#undef ZA_HF
  return za_launch_status();
}

// A decode batch's folded queries in one launch: every head's product of x's columns [0, K) into out's [0, N), and x's
// columns [K, K + Dr) rotated into out's [N, N + Dr), to the bits of za_head_linear and za_rotate_part, whose second
// launch took 4 us of a layer (8 rows of 16 heads).  At most 16 tokens, bfloat16, K below HL_SPLIT_MIN_K.
extern "C" int za_latent_fold(const void* x, int x_ld, const void* W, void* out, int o_ld, int n_tokens, int heads, int N,
                              int K, int Dr, const int* positions, const float* inv_freq, int rot_dims, int adjacent,
                              float magnitude, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  if (n_tokens < 0 || heads <= 0 || heads > 65535 || N <= 0 || K <= 0 || Dr <= 0 || rot_dims < 0 || rot_dims > Dr ||
      rot_dims % 2 || !x || !W || !out || K + Dr > x_ld || N + Dr > o_ld || (rot_dims > 0 && (!positions || !inv_freq)))
    return ZA_ERR_ARG;
  if (n_tokens > 16 || K >= HL_SPLIT_MIN_K || K % 8 || x_ld % 8 || !positions ||
      (((uintptr_t)x | (uintptr_t)W) & 15) != 0)
    return ZA_ERR_UNSUPPORTED;
  const HeadLinearArgs a{x, W, out, nullptr, n_tokens, heads, N, K, x_ld, 0, o_ld, 0, 0, 0, 0,
                         Dr, K, N, rot_dims, adjacent, magnitude, positions, inv_freq};
  hipLaunchKernelGGL((head_linear_rows16_kernel<bf16_t, false>), dim3(1, (unsigned)((N + 63) / 64) + 1, heads), dim3(256),
                     0, stream, a);
  return za_launch_status();
}

// ---------------------------------------------------------------- latent_attention
// The general kernel: any sizes, 32-bit or bfloat16 storage, everything computed in 32-bit.
// A workgroup serves one work item (up to `count` consecutive query tokens of one request)
// and one chunk of up to LA_MAX_ROWS / count heads; a tile of KT cached rows staged in LDS
// is shared by all of them.  Rows (token, head) are dealt to the four waves; in the score
// phase a lane owns a key, in the value phase it owns latent elements.  Contexts may be cut
// into `nsplit` ranges of `keys_per_split` keys, cut at key positions that depend on nothing
// else; latent_combine merges the partial (maximum, sum, accumulator).  The sink joins the
// denominator once: at the end of a whole context here, or in the merge.
#define LA_WAVES 4
#define LA_RPW 8
#define LA_MAX_ROWS (LA_WAVES * LA_RPW)
#define LA_MAX_W 576
#define LA_MAX_R 512
#define LA_RPL (LA_MAX_R / 64)        // latent elements per lane, at most

template <typename T, int KT>
__global__ void __launch_bounds__(256)
latent_attention_kernel(const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ plane,
                        long long page_stride, const int* __restrict__ block_table, int bt_stride,
                        const int* __restrict__ positions, const int* __restrict__ wi_seq,
                        const int* __restrict__ wi_row0, const int* __restrict__ wi_count,
                        float* __restrict__ part_acc, float* __restrict__ part_ml, int H, int HC,
                        int W, int R, int page_size, float scale, int keys_per_split, int nsplit,
                        const float* __restrict__ sink) {
  extern __shared__ float smem[];
  const int ldk = W + 1;
  float* Ks = smem;                       // [KT][W + 1]
  float* Qs = Ks + KT * ldk;              // [LA_MAX_ROWS][W]
  float* Ps = Qs + LA_MAX_ROWS * W;       // [LA_WAVES][64]

  const int item = blockIdx.x, z = blockIdx.z;
  const int h0 = blockIdx.y * HC;
  const int G = min(HC, H - h0);          // heads of this chunk
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int seq = wi_seq[item];
  const int row0 = wi_row0[item];
  int count = wi_count[item];
  if (count * G > LA_MAX_ROWS) count = LA_MAX_ROWS / G;   // the host never asks for more
  const int rows = count * G;
  const int* table = block_table + (size_t)seq * bt_stride;

  const int hi = positions[row0 + count - 1];   // inclusive
  int range_lo = z * keys_per_split;
  int range_hi = range_lo + keys_per_split - 1;
  if (nsplit == 1) { range_lo = 0; range_hi = hi; }
  if (range_hi > hi) range_hi = hi;

  for (int idx = tid; idx < rows * W; idx += 256) {
    const int r = idx / W, dd = idx % W;
    const int tok = row0 + r / G, h = h0 + r % G;
    Qs[r * W + dd] = to_f32<T>(q[((size_t)tok * H + h) * W + dd]);
  }

  float m[LA_RPW], l[LA_RPW], acc[LA_RPW][LA_RPL];
#pragma unroll
  for (int i = 0; i < LA_RPW; ++i) {
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int c = 0; c < LA_RPL; ++c) acc[i][c] = 0.f;
  }

  for (int tile0 = range_lo; tile0 <= range_hi; tile0 += KT) {
    __syncthreads();  // previous tile fully consumed (and Qs written, first time)
    for (int idx = tid; idx < KT * W; idx += 256) {
      const int j = idx / W, c = idx % W;
      const int kp = tile0 + j;
      float v = 0.f;
      if (kp <= range_hi) {
        const int page = table[kp / page_size];
        if (page >= 0)
          v = to_f32<T>(plane[(size_t)page * page_stride + (size_t)(kp % page_size) * W + c]);
      }
      Ks[j * ldk + c] = v;
    }
    __syncthreads();

#pragma unroll
    for (int lr = 0; lr < LA_RPW; ++lr) {
      const int r = wave + LA_WAVES * lr;
      if (r < rows) {
        const int pos = positions[row0 + r / G];
        const int kp = tile0 + lane;
        const bool valid = lane < KT && kp <= pos && kp <= range_hi;
        float s = -INFINITY;
        if (lane < KT) {
          const float* qr = Qs + r * W;
          const float* kr = Ks + lane * ldk;
          float dot = 0.f;
          for (int dd = 0; dd < W; ++dd) dot = fmaf(qr[dd], kr[dd], dot);
          if (valid) s = dot * scale;
        }
        const float tmax = wave_max(s);
        const float m_new = fmaxf(m[lr], tmax);
        if (m_new > -INFINITY) {
          const float alpha = expf(m[lr] - m_new);
          const float p = valid ? expf(s - m_new) : 0.f;
          l[lr] = l[lr] * alpha + wave_sum(p);
          m[lr] = m_new;
          __builtin_amdgcn_wave_barrier();
          Ps[wave * 64 + lane] = p;
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int c = 0; c < LA_RPL; ++c) {
            const int dd = lane + 64 * c;
            if (64 * c < R) {
              float a = acc[lr][c] * alpha;
              if (dd < R) {
#pragma unroll 8
                for (int j = 0; j < KT; ++j) a = fmaf(Ps[wave * 64 + j], Ks[j * ldk + dd], a);
              }
              acc[lr][c] = a;
            }
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
  }

#pragma unroll
  for (int lr = 0; lr < LA_RPW; ++lr) {
    const int r = wave + LA_WAVES * lr;
    if (r < rows) {
      const int tok = row0 + r / G, h = h0 + r % G;
      if (nsplit == 1) {
        if (sink) l[lr] += expf(sink[h] - m[lr]);
        const float inv = l[lr] > 0.f ? 1.0f / l[lr] : 0.f;
        T* o = out + ((size_t)tok * H + h) * R;
#pragma unroll
        for (int c = 0; c < LA_RPL; ++c) {
          const int dd = lane + 64 * c;
          if (dd < R) o[dd] = from_f32<T>(acc[lr][c] * inv);
        }
      } else {
        const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
        float* pa = part_acc + pidx * R;
#pragma unroll
        for (int c = 0; c < LA_RPL; ++c) {
          const int dd = lane + 64 * c;
          if (dd < R) pa[dd] = acc[lr][c];
        }
        if (lane == 0) {
          part_ml[pidx * 2] = m[lr];
          part_ml[pidx * 2 + 1] = l[lr];
        }
      }
    }
  }
}

// ------------------------------------------------------------ latent_attention_mfma
// bfloat16 on the matrix cores, rows of W and latents of R elements that are multiples of 8
// (16-byte pieces).  Per tile of 32 keys:
//   staging  every thread fetches, for 8 keys, the same 8 latent elements (eight 16-byte
//            loads), stores them as they are into Ks [32][W] and, turned round in its
//            registers, into Vt [R][32]: the second product wants, for one latent element,
//            consecutive keys side by side.  The rotated key part goes into Ks only.  The
//            loads of the next tile are issued before the products of this one.
//   S^T = K Q^T   keys are the rows of the first operand, 16 query rows the columns: a lane
//            ends up with ONE query row's scores for keys kq*4 .. +3 of each half of the
//            tile (kq = lane / 16)
//   p = 2^(s * scale * log2(e) - m) in 32-bit, the running maximum shared by the four lanes
//            of a query row; p is rounded to bfloat16 and the sum that normalises the result
//            is the sum of the rounded values
//   O^T += V^T P^T   P^T goes from the accumulator registers straight into the second
//            operand: the matrix core does not care how the 32 keys of a step are numbered
//            as long as both operands agree, so Vt holds, for lane group kq, the keys
//            kq*4 .. +3 and 16 + kq*4 .. +3 side by side at columns kq*8 .. +7
// Two kernels share this.  latent_attention_mfma_kernel: a workgroup of four waves serves
// one work item and one chunk of heads, at most 64 rows (token, head), 16 a wave.
// latent_decode_mfma_kernel: work items of at most 16 rows (single tokens times a chunk of
// 16 heads) that all four waves share: a wave takes every fourth 32-element step of the
// first product (the partial scores are added up through LDS, in a fixed order, so every
// wave holds the same scores) and every fourth 16-element tile of the result.
// Ranges of keys (`nsplit` > 1) leave (maximum on the natural scale, sum, accumulator) for
// latent_combine; the sink joins the denominator once, here or there.
// WS, RT: the most 32-element steps of a row and 16-element tiles of the latent that an
// instance holds in registers.
#define LM_KT 32
#define LM_VS (LM_KT + 8)
#define LM_NT 256
// Vt holds latent element e at row (e % 8) * P + e / 8, P = lm_vp(tiles of 16 elements): the
// threads of a wave store eight neighbouring rows each, at neighbouring e / 8, and a fragment
// reads 16 neighbouring e; with P = 2 (mod 16) and rows of 80 bytes neither meets a bank twice.
__host__ __device__ __forceinline__ int lm_vp(int rt) { return (2 * rt - 2 + 15) / 16 * 16 + 2; }
#define LM_LOG2E 1.4426950408889634f
#define LM_LN2 0.6931471805599453f

struct LmTile {
  bf16x8_t a[8];   // 8 keys x the same 8 latent elements
  bf16x8_t rot;    // 8 elements of one key's rotated part
};

struct LmCache {
  const bf16_t* plane;
  long long page_stride;
  const int* table;
  int page_size, shift;   // shift: log2(page_size), or -1
  int W, R;
};

// The page of key position `kp` (clamped into the range, so the entry exists) and the key's
// place in it: loads that depend on nothing but the tile, issued for all keys at once.
__device__ __forceinline__ int lm_page(const LmCache& c, int kp, int& off) {
  if (c.shift >= 0) {
    off = kp & (c.page_size - 1);
    return c.table[kp >> c.shift];
  }
  off = kp % c.page_size;
  return c.table[kp / c.page_size];
}

// Key `j` of the eight that lane group `g` feeds the second product side by side.
__device__ __forceinline__ int lm_key(int g, int j) { return j < 4 ? g * 4 + j : 16 + g * 4 + (j - 4); }

// No branch between the loads: a key beyond the range reads the range's last key, a page
// that is not there reads page 0, and the value is dropped afterwards.
__device__ __forceinline__ void lm_fetch(LmTile& t, const LmCache& c, int tile0, int range_hi, int tid) {
  const int nchunk = c.R / 8, rchunk = (c.W - c.R) / 8;
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  if (tid < 4 * nchunk) {          // R <= 512: a block a thread at most
    const int ch = tid % nchunk, g = tid / nchunk;
    int page[8], off[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) page[j] = lm_page(c, min(tile0 + lm_key(g, j), range_hi), off[j]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      t.a[j] = *reinterpret_cast<const bf16x8_t*>(
          c.plane + (size_t)max(page[j], 0) * c.page_stride + (size_t)off[j] * c.W + ch * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (tile0 + lm_key(g, j) > range_hi || page[j] < 0) t.a[j] = zero8;
  }
  t.rot = zero8;
  if (tid < LM_KT * rchunk) {
    const int kp = tile0 + tid / rchunk;
    int off;
    const int page = lm_page(c, min(kp, range_hi), off);
    const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(
        c.plane + (size_t)max(page, 0) * c.page_stride + (size_t)off * c.W + c.R + (tid % rchunk) * 8);
    if (kp <= range_hi && page >= 0) t.rot = v;
  }
}

__device__ __forceinline__ void lm_store(const LmTile& t, const LmCache& c, bf16_t* Ks, bf16_t* Vt,
                                         int KS, int VP, int tile0, int range_hi, int tid) {
  const int nchunk = c.R / 8, rchunk = (c.W - c.R) / 8;
  if (tid < 4 * nchunk) {
    const int ch = tid % nchunk, g = tid / nchunk;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<bf16x8_t*>(Ks + lm_key(g, j) * KS + ch * 8) = t.a[j];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      bf16x8_t v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = t.a[j][r];
      *reinterpret_cast<bf16x8_t*>(Vt + (r * VP + ch) * LM_VS + g * 8) = v;
    }
  }
  if (tid < LM_KT * rchunk)
    *reinterpret_cast<bf16x8_t*>(Ks + (tid / rchunk) * KS + c.R + (tid % rchunk) * 8) = t.rot;
  // a rotated part of more than 64 elements: the rest, not fetched ahead
  for (int i = tid + LM_NT; i < LM_KT * rchunk; i += LM_NT) {
    const int key = i / rchunk, kp = tile0 + key;
    bf16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (kp <= range_hi) {
      int off;
      const int page = lm_page(c, kp, off);
      if (page >= 0)
        v = *reinterpret_cast<const bf16x8_t*>(c.plane + (size_t)page * c.page_stride +
                                               (size_t)off * c.W + c.R + (i % rchunk) * 8);
    }
    *reinterpret_cast<bf16x8_t*>(Ks + key * KS + c.R + (i % rchunk) * 8) = v;
  }
}

// One query row's scores of a tile (this lane's eight keys) -> its probabilities as the
// second operand's fragment; updates the running maximum and sum; returns the factor the
// accumulator takes.
__device__ __forceinline__ float lm_softmax(const f32x4_t& s0, const f32x4_t& s1, int tile0, int kq,
                                            int pos_q, int range_hi, float scale_log2, float& m,
                                            float& l, bf16x8_t& pf) {
  float sc[8];
  float tmax = -INFINITY;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int kp = tile0 + lm_key(kq, i);
    const float v = (i < 4 ? s0[i] : s1[i - 4]) * scale_log2;
    sc[i] = (kp <= pos_q && kp <= range_hi) ? v : -INFINITY;
    tmax = fmaxf(tmax, sc[i]);
  }
  tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
  tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
  const float m_new = fmaxf(m, tmax);
  const float m_use = m_new > -INFINITY ? m_new : 0.f;
  const float alpha = m == m_new ? 1.0f : exp2f(m - m_use);
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bf16_t pb = (bf16_t)exp2f(sc[i] - m_use);
    pf[i] = pb;
    psum += (float)pb;
  }
  l = l * alpha + psum;
  m = m_new;
  return alpha;
}

template <int WS, int RT>
__global__ void __launch_bounds__(LM_NT)
latent_attention_mfma_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out,
                             const bf16_t* __restrict__ plane, long long page_stride,
                             const int* __restrict__ block_table, int bt_stride,
                             const int* __restrict__ positions, const int* __restrict__ wi_seq,
                             const int* __restrict__ wi_row0, const int* __restrict__ wi_count,
                             float* __restrict__ part_acc, float* __restrict__ part_ml, int H,
                             int HC, int W, int R, int page_size, int page_shift,
                             float scale_log2, int keys_per_split, int nsplit,
                             const float* __restrict__ sink) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lm_lds[];
  const int ws = (W + 31) / 32, rt = (R + 15) / 16;
  const int KS = ws * 32 + 8;                       // elements from row to row of Ks
  bf16_t* Ks = reinterpret_cast<bf16_t*>(lm_lds);   // [LM_KT][KS]
  bf16_t* Vt = Ks + LM_KT * KS;                     // [8 * VP][LM_VS]
  const int VP = lm_vp(rt);

  // the last items first: within a request the later an item, the more keys it has, and
  // workgroups start in the order of their numbers, so the long ones do not start last
  const int item = gridDim.x - 1 - blockIdx.x, z = blockIdx.z;
  const int h0 = blockIdx.y * HC;
  const int G = min(HC, H - h0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kq = lane >> 4;
  const int seq = wi_seq[item];
  const int row0 = wi_row0[item];
  int count = wi_count[item];
  if (count * G > 64) count = 64 / G;               // the host never asks for more
  const int rows = count * G;
  const int hi = positions[row0 + count - 1];       // inclusive
  int range_lo = z * keys_per_split;
  int range_hi = range_lo + keys_per_split - 1;
  if (nsplit == 1) { range_lo = 0; range_hi = hi; }
  if (range_hi > hi) range_hi = hi;
  const LmCache cache = {plane, page_stride, block_table + (size_t)seq * bt_stride, page_size,
                         page_shift, W, R};

  // columns of Ks beyond W and rows of Vt beyond R stay zero: clear everything once
  {
    const int words = (LM_KT * KS + 8 * VP * LM_VS) / 2;
    uint32_t* w = reinterpret_cast<uint32_t*>(lm_lds);
    for (int i = tid; i < words; i += LM_NT) w[i] = 0u;
  }

  const int my = wave * 16 + r16;
  const bool row_ok = my < rows;
  const bool wave_on = wave * 16 < rows;
  const int tok = row0 + (row_ok ? my / G : 0);
  const int h = h0 + (row_ok ? my % G : 0);
  const int pos_q = row_ok ? positions[tok] : -1;
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_t qf[WS];
#pragma unroll
  for (int ks = 0; ks < WS; ++ks) {
    const int c = ks * 32 + kq * 8;
    qf[ks] = (row_ok && c < W)
                 ? *reinterpret_cast<const bf16x8_t*>(q + ((size_t)tok * H + h) * W + c)
                 : zero8;
  }
  float m = -INFINITY, l = 0.f;
  f32x4_t o[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  LmTile regs;
  if (range_lo <= range_hi) lm_fetch(regs, cache, range_lo, range_hi, tid);
  for (int tile0 = range_lo; tile0 <= range_hi; tile0 += LM_KT) {
    __syncthreads();      // the tile before is used up (first time: the clearing is done)
    lm_store(regs, cache, Ks, Vt, KS, VP, tile0, range_hi, tid);
    __syncthreads();
    if (tile0 + LM_KT <= range_hi) lm_fetch(regs, cache, tile0 + LM_KT, range_hi, tid);
    if (wave_on) {
      f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < WS; ++ks) {
        if (ks < ws) {
          const bf16x8_t k0 =
              *reinterpret_cast<const bf16x8_t*>(Ks + r16 * KS + ks * 32 + kq * 8);
          const bf16x8_t k1 =
              *reinterpret_cast<const bf16x8_t*>(Ks + (16 + r16) * KS + ks * 32 + kq * 8);
          s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[ks], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[ks], s1, 0, 0, 0);
        }
      }
      bf16x8_t pf;
      const float alpha = lm_softmax(s0, s1, tile0, kq, pos_q, range_hi, scale_log2, m, l, pf);
      if (!__all(alpha == 1.0f)) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if (t < rt) { o[t][0] *= alpha; o[t][1] *= alpha; o[t][2] *= alpha; o[t][3] *= alpha; }
        }
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        if (t < rt) {
          const bf16x8_t vf = *reinterpret_cast<const bf16x8_t*>(
              Vt + ((r16 & 7) * VP + 2 * t + (r16 >> 3)) * LM_VS + kq * 8);
          o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[t], 0, 0, 0);
        }
      }
    }
  }

  if (!wave_on) return;
  float lt = l;
  lt += __shfl_xor(lt, 16, 64);
  lt += __shfl_xor(lt, 32, 64);
  if (!row_ok) return;
  if (nsplit == 1) {
    if (sink) lt += exp2f(sink[h] * LM_LOG2E - m);
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    bf16_t* orow = out + ((size_t)tok * H + h) * R;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int r = t * 16 + kq * 4;
      if (t < rt && r < R) {
        bf16x4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(o[t][i] * inv);
        *reinterpret_cast<bf16x4_t*>(orow + r) = v;
      }
    }
  } else {
    const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
    float* pa = part_acc + pidx * R;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int r = t * 16 + kq * 4;
      if (t < rt && r < R) *reinterpret_cast<f32x4_t*>(pa + r) = o[t];
    }
    if (kq == 0) {
      part_ml[pidx * 2] = m * LM_LN2;
      part_ml[pidx * 2 + 1] = lt;
    }
  }
}

// ------------------------------------------------------------ latent_prefill_mfma
// The same for prompt portions and mixed steps where R is 128, 256 or 512 and the rotated part
// 0, 32 or 64: eight waves serve one work item and one chunk of heads, at most 64 rows, 64 keys
// a tile, and every fragment serves all the rows that it can.
//   tiles    go from memory into one of two places in LDS without passing registers, a wave
//            eight keys, the next tile while this one is used.  A key's 16-byte pieces lie in
//            the order piece ^ (key % 8), so that neither kind of read meets a bank twice.
//   S^T      wave w takes the 16 keys w % 4 and 32 rows (w / 4): a fragment of keys serves two
//            products, and the rows stay in registers
//   softmax  the waves' maxima meet in LDS; every wave then holds every row's maximum, and
//            leaves its probabilities (bfloat16) in LDS
//   O^T      wave w takes R / 8 of the latent for all 64 rows: the tile's keys are read turned
//            round (ds_read_b64_tr_b16: of 4 keys x 16 elements a lane gets one element's four
//            keys), each once a workgroup
// Reads of LDS and matrix products would bound it in equal parts (35 fragments for 68 products a
// wave and tile at R = 512 with 64 rotated); what does are the waits between them, three meetings
// of the waves a tile.  (Four waves that each take 16 rows through the whole tile, as below for
// other widths, read a fragment for every product and wait for each, one wave a SIMD.)
// 16 heads, a first portion of 1,777 tokens, R = 512 with 64 rotated: 115 us against 313 of that
// form, R = 256: 84 against 191, R = 128: 71 against 147; 8 tokens behind 2,048 cached ones beside
// 256 new ones 68 against 99; 40 tokens of 4 heads 18 against 20.  Its error against 64 bits is the
// same (1.85e-3 of the result's norm, the rounding of probabilities and result).
#define LP_KT 64
#define LP_NT 512
#define LP_PAIRS 2          // pairs of fragments that a wave takes at once (3: registers run over)

// The waits are written by hand: the compiler would wait for the next tile's requests before
// any read of LDS.
__device__ __forceinline__ void lp_meet() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Fragments 2 * PAIRS from two addresses, 128 bytes from pair to pair.
template <int PAIRS>
__device__ __forceinline__ void lp_take_keys(bf16x8_t (&f)[2 * LP_PAIRS], unsigned even, unsigned odd) {
  static_assert(PAIRS == 1 || PAIRS == LP_PAIRS, "the forms below");
  if constexpr (PAIRS == 2)
    asm volatile(
        "ds_read_b128 %0, %4 offset:0\n" "ds_read_b128 %1, %5 offset:0\n"
        "ds_read_b128 %2, %4 offset:128\n" "ds_read_b128 %3, %5 offset:128\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
        : "v"(even), "v"(odd)
        : "memory");
  if constexpr (PAIRS == 1)
    asm volatile(
        "ds_read_b128 %0, %2 offset:0\n" "ds_read_b128 %1, %3 offset:0\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0]), "=&v"(f[1])
        : "v"(even), "v"(odd)
        : "memory");
}

// Of 32 keys: the probabilities of four times 16 rows and the first one or two tiles of the
// latent (from two addresses each), or the next two tiles alone.
template <int TILES, bool P>
__device__ __forceinline__ void lp_take_values(bf16x8_t (&p)[4], bf16x4_t (&v)[TILES][2], unsigned pa,
                                               const unsigned (&va)[TILES][2]) {
  if constexpr (TILES == 2 && P)
    asm volatile(
        "ds_read_b128 %0, %8 offset:0\n" "ds_read_b128 %1, %8 offset:2048\n"
        "ds_read_b128 %2, %8 offset:4096\n" "ds_read_b128 %3, %8 offset:6144\n"
        "ds_read_b64_tr_b16 %4, %9\n" "ds_read_b64_tr_b16 %5, %10\n"
        "ds_read_b64_tr_b16 %6, %11\n" "ds_read_b64_tr_b16 %7, %12\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3]), "=&v"(v[0][0]), "=&v"(v[0][1]),
          "=&v"(v[1][0]), "=&v"(v[1][1])
        : "v"(pa), "v"(va[0][0]), "v"(va[0][1]), "v"(va[1][0]), "v"(va[1][1])
        : "memory");
  if constexpr (TILES == 2 && !P)
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4\n" "ds_read_b64_tr_b16 %1, %5\n"
        "ds_read_b64_tr_b16 %2, %6\n" "ds_read_b64_tr_b16 %3, %7\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1])
        : "v"(va[0][0]), "v"(va[0][1]), "v"(va[1][0]), "v"(va[1][1])
        : "memory");
  if constexpr (TILES == 1)
    asm volatile(
        "ds_read_b128 %0, %6 offset:0\n" "ds_read_b128 %1, %6 offset:2048\n"
        "ds_read_b128 %2, %6 offset:4096\n" "ds_read_b128 %3, %6 offset:6144\n"
        "ds_read_b64_tr_b16 %4, %7\n" "ds_read_b64_tr_b16 %5, %8\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3]), "=&v"(v[0][0]), "=&v"(v[0][1])
        : "v"(pa), "v"(va[0][0]), "v"(va[0][1])
        : "memory");
}

template <int RT, int DT>
struct LpShape {
  static constexpr int R = RT * 16, W = R + DT * 32, WS = W / 32;
  static constexpr int PIECES = (WS * 4 + 7) / 8 * 8;      // of a key in LDS
  static constexpr int TILE = LP_KT * PIECES * 8;          // elements of a place
  static constexpr int KEPT = WS < 17 ? WS : 17;           // steps of the rows in registers; the rest in LDS
  static constexpr size_t LDS = (size_t)2 * TILE * 2 + 64 * LP_KT * 2 + 64 * 4 * 4 + (WS - KEPT) * 64 * 32 * 2;
};

// What a key without a page (an entry below zero) holds; the requests into LDS have no other zeros.
__device__ __attribute__((aligned(16))) bf16_t lp_no_row[512 + 64];

template <int RT, int DT>
__global__ void __launch_bounds__(LP_NT)
latent_prefill_mfma_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out,
                           const bf16_t* __restrict__ plane, long long page_stride,
                           const int* __restrict__ block_table, int bt_stride,
                           const int* __restrict__ positions, const int* __restrict__ wi_seq,
                           const int* __restrict__ wi_row0, const int* __restrict__ wi_count,
                           float* __restrict__ part_acc, float* __restrict__ part_ml, int H,
                           int HC, int page_shift, float scale_log2,
                           int keys_per_split, int nsplit, const float* __restrict__ sink) {
  using S = LpShape<RT, DT>;
  constexpr int R = S::R, W = S::W, WS = S::WS, NP = S::PIECES, OT = RT / 8, KEPT = S::KEPT;
  static_assert(WS - KEPT <= 1, "one step of the rows in LDS at most");
  extern __shared__ __attribute__((aligned(16))) unsigned char lm_lds[];
  bf16_t* Ks = reinterpret_cast<bf16_t*>(lm_lds);                 // [2][LP_KT][NP * 8]
  bf16_t* Ps = Ks + 2 * S::TILE;                                  // [64 rows][LP_KT]
  float* Xs = reinterpret_cast<float*>(Ps + 64 * LP_KT);          // [64 rows][4]
  bf16_t* Qs = reinterpret_cast<bf16_t*>(Xs + 64 * 4);            // [4][64 lanes][8]: the rows' last step

  // the last items first: within a request the later an item, the more keys it has, and
  // workgroups start in the order of their numbers, so the long ones do not start last
  const int item = gridDim.x - 1 - blockIdx.x, z = blockIdx.z;
  const int h0 = blockIdx.y * HC;
  const int G = min(HC, H - h0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int kt = wave & 3, rh = wave >> 2;
  const int seq = wi_seq[item];
  const int row0 = wi_row0[item];
  int count = wi_count[item];
  if (count * G > 64) count = 64 / G;               // the host never asks for more
  const int rows = count * G;
  const int hi = positions[row0 + count - 1];       // inclusive
  int range_lo = z * keys_per_split;
  int range_hi = range_lo + keys_per_split - 1;
  if (nsplit == 1) { range_lo = 0; range_hi = hi; }
  if (range_hi > hi) range_hi = hi;
  const int* table = block_table + (size_t)seq * bt_stride;

  // the page of key wave * 8 + lane % 8 of a tile (a key beyond the range reads the range's last
  // one, whose scores are then masked)
  auto page_of = [&](int tile0) -> int {
    const int kp = min(tile0 + wave * 8 + (lane & 7), range_hi);
    return table[kp >> page_shift];
  };
  auto request = [&](int page, int tile0, int buffer) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                  // (worked out again for each tile: registers)
    const int kp = min(tile0 + wave * 8 + (lane & 7), range_hi);
    const int off = kp & ((1 << page_shift) - 1);
    const long long at = (long long)(page >= 0 ? plane + (long long)page * page_stride + (long long)off * W
                                               : (const bf16_t*)lp_no_row);
    long long base[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      base[j] = (long long)((unsigned)__builtin_amdgcn_readlane((int)at, j)) |
                ((long long)__builtin_amdgcn_readlane((int)(at >> 32), j) << 32);
    bf16_t* to = Ks + buffer * S::TILE + wave * 8 * NP * 8;
#pragma unroll
    for (int i = 0; i < NP / 8; ++i) {
      long long from = base[i * 64 / NP];
      int key = i * 64 / NP;
#pragma unroll
      for (int j = i * 64 / NP + 1; j <= (i * 64 + 63) / NP; ++j)
        if (lane >= j * NP - i * 64) { from = base[j]; key = j; }
      int piece = (i * 64 + lane - key * NP) ^ key;
      if (WS % 2 && piece >= W / 8) piece = 0;       // room that no fragment reads
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)((const bf16_t*)from + piece * 8),
          (__attribute__((address_space(3))) void*)(to + i * 512), 16, 0, 0);
    }
  };

  int page = 0;                // of the tile that is requested next
  if (range_lo <= range_hi) {
    request(page_of(range_lo), range_lo, 0);
    page = page_of(range_lo + LP_KT);
  }

  // this wave's rows of the first product
  bf16x8_t qf[2][KEPT];
  int pos_q[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int my = (rh * 2 + a) * 16 + r16;
    const bool row_ok = my < rows;
    const int tok = row0 + (row_ok ? my / G : 0), h = h0 + (row_ok ? my % G : 0);
    pos_q[a] = row_ok ? positions[tok] : -1;
    const bf16_t* qrow = q + ((size_t)tok * H + h) * W + kq * 8;     // (a row beyond: masked below)
#pragma unroll
    for (int ks = 0; ks < KEPT; ++ks) qf[a][ks] = *reinterpret_cast<const bf16x8_t*>(qrow + ks * 32);
    if (KEPT < WS && kt == 0) {
      const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(qrow + KEPT * 32);
      asm volatile("ds_write_b128 %0, %1" ::"v"(lds_address(Qs) + (rh * 2 + a) * 1024 + lane * 16), "v"(v) : "memory");
    }
  }
  float m[4], l[2] = {0.f, 0.f};
  f32x4_t o[4][OT];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    m[a] = -INFINITY;
#pragma unroll
    for (int t = 0; t < OT; ++t) o[a][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const unsigned ks_at = lds_address(Ks), ps_at = lds_address(Ps), xs_at = lds_address(Xs);
  int buffer = 0;
  for (int tile0 = range_lo; tile0 <= range_hi; tile0 += LP_KT, buffer ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lp_meet();            // this tile is here, and nobody reads the other place any more
    if (tile0 + LP_KT <= range_hi) {
      request(page, tile0 + LP_KT, buffer ^ 1);
      page = page_of(tile0 + 2 * LP_KT);
    }
    const unsigned in_buffer = buffer * S::TILE * 2;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int r16 = lane & 15, kq = lane >> 4;
    const unsigned key_row = ks_at + (kt * 16 + r16) * NP * 16 + in_buffer;
    const unsigned even = key_row + ((kq ^ (r16 & 7)) << 4), odd = even ^ 64;
    f32x4_t s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int PAIRS = (WS + 1) / 2;
#pragma unroll
    for (int b = 0; b < PAIRS; b += LP_PAIRS) {
      bf16x8_t kf[2 * LP_PAIRS];
      if (b + LP_PAIRS <= PAIRS) lp_take_keys<LP_PAIRS>(kf, even + b * 128, odd + b * 128);
      else lp_take_keys<1>(kf, even + b * 128, odd + b * 128);
#pragma unroll
      for (int i = 0; i < 2 * LP_PAIRS; ++i) {
        const int ks = b * 2 + i;
        if (KEPT < WS && ks == KEPT) {
          bf16x8_t qs[2];
          asm volatile("ds_read_b128 %0, %2\n" "ds_read_b128 %1, %2 offset:1024\n" "s_waitcnt lgkmcnt(0)"
                       : "=&v"(qs[0]), "=&v"(qs[1])
                       : "v"(lds_address(Qs) + rh * 2048 + lane * 16)
                       : "memory");
          s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i], qs[0], s[0], 0, 0, 0);
          s[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i], qs[1], s[1], 0, 0, 0);
        } else if (ks < KEPT) {
          s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i], qf[0][ks], s[0], 0, 0, 0);
          s[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i], qf[1][ks], s[1], 0, 0, 0);
        }
      }
    }
    float top[2];
    const int kp0 = tile0 + kt * 16 + kq * 4;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      top[a] = -INFINITY;
      const int last = min(pos_q[a], range_hi);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[a][i] = kp0 + i <= last ? s[a][i] * scale_log2 : -INFINITY;
        top[a] = fmaxf(top[a], s[a][i]);
      }
      top[a] = fmaxf(top[a], __shfl_xor(top[a], 16, 64));
      top[a] = fmaxf(top[a], __shfl_xor(top[a], 32, 64));
    }
    if (kq < 2)
      asm volatile("ds_write_b32 %0, %1" ::"v"(xs_at + (((rh * 2 + kq) * 16 + r16) * 4 + kt) * 4),
                   "v"(kq ? top[1] : top[0]) : "memory");
    lp_meet();
    float alpha[4];
#pragma unroll
    for (int b = 0; b < 4; b += 2) {
      f32x4_t seen[2];
      asm volatile("ds_read_b128 %0, %2\n" "ds_read_b128 %1, %2 offset:256\n" "s_waitcnt lgkmcnt(0)"
                   : "=&v"(seen[0]), "=&v"(seen[1])
                   : "v"(xs_at + r16 * 16 + b * 256)
                   : "memory");
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int a = b + i;
        const float m_new = fmaxf(fmaxf(fmaxf(seen[i][0], seen[i][1]), fmaxf(seen[i][2], seen[i][3])), m[a]);
        alpha[a] = m[a] == m_new ? 1.0f : exp2f(m[a] - m_new);
        m[a] = m_new;
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float mx = rh ? m[2 + a] : m[a];
      const float m_use = mx > -INFINITY ? mx : 0.f;
      bf16x4_t pb;
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pb[i] = (bf16_t)exp2f(s[a][i] - m_use);
        psum += (float)pb[i];
      }
      l[a] = l[a] * (rh ? alpha[2 + a] : alpha[a]) + psum;
      asm volatile("ds_write_b64 %0, %1" ::"v"(ps_at + ((rh * 2 + a) * 16 + r16) * (LP_KT * 2) +
                                               (((kt * 2 + (kq >> 1)) ^ (r16 & 7)) << 4) + (kq & 1) * 8),
                   "v"(pb) : "memory");
    }
    lp_meet();
    if (!__all(alpha[0] == 1.0f && alpha[1] == 1.0f && alpha[2] == 1.0f && alpha[3] == 1.0f)) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int t = 0; t < OT; ++t) {
          o[a][t][0] *= alpha[a]; o[a][t][1] *= alpha[a];
          o[a][t][2] *= alpha[a]; o[a][t][3] *= alpha[a];
        }
    }
#pragma unroll
    for (int step = 0; step < LP_KT / 32; ++step) {
      int lane = threadIdx.x & 63;
      asm volatile("" : "+v"(lane));
      const int r16 = lane & 15, kq = lane >> 4;
      constexpr int TILES = OT < 2 ? OT : 2;
      bf16x8_t pf[4];
#pragma unroll
      for (int t0 = 0; t0 < OT; t0 += TILES) {
        unsigned va[TILES][2];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            const int low = hf * 4 + (r16 >> 2);         // of the key that this lane points at
            const int piece = (wave * OT + t0 + t) * 2 + ((r16 >> 1) & 1);
            va[t][hf] = ks_at + in_buffer + (step * 32 + kq * 8 + low) * NP * 16 + ((piece ^ low) << 4) +
                        (r16 & 1) * 8;
          }
        bf16x4_t vh[TILES][2];
        const unsigned pa = ps_at + r16 * (LP_KT * 2) + (((step * 4 + kq) ^ (r16 & 7)) << 4);
        if (t0 == 0) lp_take_values<TILES, true>(pf, vh, pa, va);
        else lp_take_values<TILES, false>(pf, vh, pa, va);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
          const bf16x8_t vf = __builtin_shufflevector(vh[t][0], vh[t][1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int a = 0; a < 4; ++a)
            o[a][t0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[a], o[a][t0 + t], 0, 0, 0);
        }
      }
    }
  }

  // the rows' sums meet like their maxima
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    l[a] += __shfl_xor(l[a], 16, 64);
    l[a] += __shfl_xor(l[a], 32, 64);
  }
  __syncthreads();
  if (kq < 2) Xs[((rh * 2 + kq) * 16 + r16) * 4 + kt] = kq ? l[1] : l[0];
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int my = a * 16 + r16;
    if (my >= rows) continue;
    const int tok = row0 + my / G, h = h0 + my % G;
    const f32x4_t part = *reinterpret_cast<const f32x4_t*>(Xs + my * 4);
    float lt = (part[0] + part[1]) + (part[2] + part[3]);
    const int e = wave * OT * 16 + kq * 4;
    if (nsplit == 1) {
      if (sink) lt += exp2f(sink[h] * LM_LOG2E - m[a]);
      const float inv = lt > 0.f ? 1.0f / lt : 0.f;
      bf16_t* orow = out + ((size_t)tok * H + h) * R + e;
#pragma unroll
      for (int t = 0; t < OT; ++t) {
        bf16x4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(o[a][t][i] * inv);
        *reinterpret_cast<bf16x4_t*>(orow + t * 16) = v;
      }
    } else {
      const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
      float* pa = part_acc + pidx * R + e;
#pragma unroll
      for (int t = 0; t < OT; ++t) *reinterpret_cast<f32x4_t*>(pa + t * 16) = o[a][t];
      if (wave == 0 && kq == 0) {
        part_ml[pidx * 2] = m[a] * LM_LN2;
        part_ml[pidx * 2 + 1] = lt;
      }
    }
  }
}

template <int WS, int RT>
__global__ void __launch_bounds__(LM_NT)
latent_decode_mfma_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out,
                          const bf16_t* __restrict__ plane, long long page_stride,
                          const int* __restrict__ block_table, int bt_stride,
                          const int* __restrict__ positions, const int* __restrict__ wi_seq,
                          const int* __restrict__ wi_row0, const int* __restrict__ wi_count,
                          float* __restrict__ part_acc, float* __restrict__ part_ml, int H, int HC,
                          int W, int R, int page_size, int page_shift, float scale_log2,
                          int keys_per_split, int nsplit, const float* __restrict__ sink) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lm_lds[];
  constexpr int QW = (WS + 3) / 4, OT = (RT + 3) / 4;
  const int ws = (W + 31) / 32, rt = (R + 15) / 16;
  const int KS = ws * 32 + 8;
  bf16_t* Ks = reinterpret_cast<bf16_t*>(lm_lds);   // [LM_KT][KS]
  bf16_t* Vt = Ks + LM_KT * KS;                     // [8 * VP][LM_VS]
  const int VP = lm_vp(rt);
  float* Sx = reinterpret_cast<float*>(Vt + 8 * lm_vp(rt) * LM_VS);   // [4 waves][64 lanes][8]

  const int item = blockIdx.x, z = blockIdx.z;
  const int h0 = blockIdx.y * HC;
  const int G = min(HC, H - h0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kq = lane >> 4;
  const int seq = wi_seq[item];
  const int row0 = wi_row0[item];
  int count = wi_count[item];
  if (count * G > 16) count = 16 / G;               // the host never asks for more
  const int rows = count * G;
  const int hi = positions[row0 + count - 1];       // inclusive
  int range_lo = z * keys_per_split;
  int range_hi = range_lo + keys_per_split - 1;
  if (nsplit == 1) { range_lo = 0; range_hi = hi; }
  if (range_hi > hi) range_hi = hi;
  const LmCache cache = {plane, page_stride, block_table + (size_t)seq * bt_stride, page_size,
                         page_shift, W, R};
  const bool row_ok = r16 < rows;
  const int tok = row0 + (row_ok ? r16 / G : 0);
  const int h = h0 + (row_ok ? r16 % G : 0);
  if (nsplit > 1 && range_lo > hi) {
    // a range behind the context (a recorded step is cut for the longest of its kind): no result, which
    // a sum of -1 says
    if (row_ok && wave == 0 && kq == 0) {
      const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
      part_ml[pidx * 2] = -INFINITY;
      part_ml[pidx * 2 + 1] = -1.f;
    }
    return;
  }
  LmTile regs_a, regs_b;
  if (range_lo <= range_hi) lm_fetch(regs_a, cache, range_lo, range_hi, tid);
  if (range_lo + LM_KT <= range_hi) lm_fetch(regs_b, cache, range_lo + LM_KT, range_hi, tid);
  // (what a row has beyond whole steps and tiles; without such a rest all that is read is stored first)
  if (W % 32 || R % 16) {
    const int words = (LM_KT * KS + 8 * VP * LM_VS) / 2;
    uint32_t* w = reinterpret_cast<uint32_t*>(lm_lds);
    for (int i = tid; i < words; i += LM_NT) w[i] = 0u;
  }

  const int pos_q = row_ok ? positions[tok] : -1;
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8_t qf[QW];          // the steps wave, wave + 4, ... of the row
#pragma unroll
  for (int j = 0; j < QW; ++j) {
    const int c = (j * 4 + wave) * 32 + kq * 8;
    qf[j] = (row_ok && c < W)
                ? *reinterpret_cast<const bf16x8_t*>(q + ((size_t)tok * H + h) * W + c)
                : zero8;
  }
  float m = -INFINITY, l = 0.f;
  f32x4_t o[OT];            // the tiles wave, wave + 4, ... of the result
#pragma unroll
  for (int j = 0; j < OT; ++j) o[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // two tiles are on their way while one is worked on: a step of few rows has little to do
  // a tile, and what it waits for is memory
  auto tile = [&](LmTile& regs, int tile0) {
    __syncthreads();
    lm_store(regs, cache, Ks, Vt, KS, VP, tile0, range_hi, tid);
    __syncthreads();
    if (tile0 + 2 * LM_KT <= range_hi) lm_fetch(regs, cache, tile0 + 2 * LM_KT, range_hi, tid);
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < QW; ++j) {
      const int ks = j * 4 + wave;
      if (ks < ws) {
        const bf16x8_t k0 = *reinterpret_cast<const bf16x8_t*>(Ks + r16 * KS + ks * 32 + kq * 8);
        const bf16x8_t k1 =
            *reinterpret_cast<const bf16x8_t*>(Ks + (16 + r16) * KS + ks * 32 + kq * 8);
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[j], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[j], s1, 0, 0, 0);
      }
    }
    *reinterpret_cast<f32x4_t*>(Sx + (wave * 64 + lane) * 8) = s0;
    *reinterpret_cast<f32x4_t*>(Sx + (wave * 64 + lane) * 8 + 4) = s1;
    __syncthreads();
    s0 = *reinterpret_cast<const f32x4_t*>(Sx + lane * 8);
    s1 = *reinterpret_cast<const f32x4_t*>(Sx + lane * 8 + 4);
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(Sx + (w * 64 + lane) * 8);
      const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(Sx + (w * 64 + lane) * 8 + 4);
      s0[0] += a0[0]; s0[1] += a0[1]; s0[2] += a0[2]; s0[3] += a0[3];
      s1[0] += a1[0]; s1[1] += a1[1]; s1[2] += a1[2]; s1[3] += a1[3];
    }
    bf16x8_t pf;
    const float alpha = lm_softmax(s0, s1, tile0, kq, pos_q, range_hi, scale_log2, m, l, pf);
#pragma unroll
    for (int j = 0; j < OT; ++j) {
      const int t = j * 4 + wave;
      if (t < rt) {
        const bf16x8_t vf = *reinterpret_cast<const bf16x8_t*>(
            Vt + ((r16 & 7) * VP + 2 * t + (r16 >> 3)) * LM_VS + kq * 8);
        f32x4_t acc = o[j];
        acc[0] *= alpha; acc[1] *= alpha; acc[2] *= alpha; acc[3] *= alpha;
        o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, acc, 0, 0, 0);
      }
    }
  };
  for (int tile0 = range_lo; tile0 <= range_hi; tile0 += 2 * LM_KT) {
    tile(regs_a, tile0);
    if (tile0 + LM_KT > range_hi) break;
    tile(regs_b, tile0 + LM_KT);
  }

  float lt = l;
  lt += __shfl_xor(lt, 16, 64);
  lt += __shfl_xor(lt, 32, 64);
  if (!row_ok) return;
  if (nsplit == 1) {
    if (sink) lt += exp2f(sink[h] * LM_LOG2E - m);
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    bf16_t* orow = out + ((size_t)tok * H + h) * R;
#pragma unroll
    for (int j = 0; j < OT; ++j) {
      const int t = j * 4 + wave, r = t * 16 + kq * 4;
      if (t < rt && r < R) {
        bf16x4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(o[j][i] * inv);
        *reinterpret_cast<bf16x4_t*>(orow + r) = v;
      }
    }
  } else {
    const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
    float* pa = part_acc + pidx * R;
#pragma unroll
    for (int j = 0; j < OT; ++j) {
      const int t = j * 4 + wave, r = t * 16 + kq * 4;
      if (t < rt && r < R) *reinterpret_cast<f32x4_t*>(pa + r) = o[j];
    }
    if (wave == 0 && kq == 0) {
      part_ml[pidx * 2] = m * LM_LN2;
      part_ml[pidx * 2 + 1] = lt;
    }
  }
}

// Single tokens, rows of whole tiles: a workgroup takes LD_KT keys at a time, 16 of them a wave, for up to 16 rows
// (token, head).  All of a range's rows are requested into LDS at once, without registers, a key's 16-byte pieces in the
// order piece ^ (key % 8); a wave has the scores of its keys, over the whole of a row; the waves' maxima meet in
// LDS, then their weights, and a wave takes every eighth of the latent over all keys, turned round on the way to
// registers (ds_read_b64_tr_b16).  A weight goes into the products as two bfloat16 numbers, it and what its rounding
// leaves: in tiles of 32 keys the running maximum has more weights of exactly one, so the same weights rounded
// once here were 1 to 3 percent further from 64 bits (8 requests at 2,050 keys 1.89e-3 and 1.86e-3; so 1.66e-3, the
// rounding of the result).  What bounds it is the way to memory (item, position, page, rows) once a range: 8 requests of
// 16 heads at 2,051 keys, R = 512 with 64 rotated, ranges of 128, with the merge: 19.1 us (weights rounded once 18.9),
// tiles of 32 through registers with three meetings each 23.5; 64 at 1,200 in ranges of 512 33.3 (32.6), before in ranges
// of 128 58; 8 at 8,000 30 (29.5) and 50.
#define LD_KT 128
#define LD_NW (LD_KT / 16)
template <int RT, int DT>
struct LdShape {
  static constexpr int R = RT * 16, W = R + DT * 32, WS = W / 32;
  static constexpr int NP = (WS * 4 + 7) / 8 * 8;            // pieces of a key in LDS
  static constexpr size_t LDS = (size_t)LD_KT * NP * 16 + 2 * 16 * LD_KT * 2 + 16 * LD_NW * 4;
};

template <int RT, int DT>
__global__ void __launch_bounds__(LD_NW * 64)
latent_decode_range_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ plane,
                           long long page_stride, const int* __restrict__ block_table, int bt_stride,
                           const int* __restrict__ positions, const int* __restrict__ wi_seq,
                           const int* __restrict__ wi_row0, const int* __restrict__ wi_count,
                           float* __restrict__ part_acc, float* __restrict__ part_ml, int H, int HC, int page_shift,
                           float scale_log2, int keys_per_split, int nsplit, const float* __restrict__ sink) {
  using S = LdShape<RT, DT>;
  static_assert(RT % LD_NW == 0, "a wave takes as much of the latent as any other");
  constexpr int R = S::R, W = S::W, WS = S::WS, NP = S::NP, OT = RT / LD_NW;
  extern __shared__ __attribute__((aligned(16))) unsigned char lm_lds[];
  unsigned char* Ks = lm_lds;                                                   // [LD_KT][NP * 16 bytes]
  unsigned char* Ps = Ks + (size_t)LD_KT * NP * 16;                             // [16 rows][LD_KT]
  unsigned char* Rs = Ps + 16 * LD_KT * 2;                                      // what rounding took from them
  float* Xs = reinterpret_cast<float*>(Rs + 16 * LD_KT * 2);                    // [16 rows][LD_NW]

  const int item = blockIdx.x, z = blockIdx.z, h0 = blockIdx.y * HC;
  const int G = min(HC, H - h0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int seq = wi_seq[item], row0 = wi_row0[item];
  const int count = min(wi_count[item], max(16 / G, 1));      // (the host never asks for more)
  const int rows = count * G;
  const int hi = positions[row0 + count - 1];                 // inclusive
  int range_lo = z * keys_per_split, range_hi = range_lo + keys_per_split - 1;
  if (nsplit == 1) { range_lo = 0; range_hi = hi; }
  range_hi = min(range_hi, hi);
  const bool row_ok = r16 < rows;
  const int tok = row0 + (row_ok ? r16 / G : 0), h = h0 + (row_ok ? r16 % G : 0);
  if (nsplit > 1 && range_lo > hi) {
    // (a range behind the context, as in the kernel above)
    if (row_ok && wave == 0 && kq == 0) {
      const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
      part_ml[pidx * 2] = -INFINITY;
      part_ml[pidx * 2 + 1] = -1.f;
    }
    return;
  }
  const int* table = block_table + (size_t)seq * bt_stride;

  // the wave's sixteen keys: a lane knows where one lies (beyond the range its last key, whose score is masked)
  // (what two waves bring is left out where none of it is in the range: nobody reads it)
  auto request = [&](int tile0) {
    if (tile0 + (wave & ~1) * 16 > range_hi) return;
    const int kp = min(tile0 + wave * 16 + r16, range_hi), page = table[kp >> page_shift];
    const bf16_t* row = page >= 0 ? plane + (long long)page * page_stride + (long long)(kp & ((1 << page_shift) - 1)) * W
                                  : (const bf16_t*)lp_no_row;
    const int low = (int)(uintptr_t)row, high = (int)((uintptr_t)row >> 32);
    unsigned char* to = Ks + wave * 16 * NP * 16;
#pragma unroll
    for (int i = 0; i < NP / 4; ++i) {
      const int at = i * 64 + lane, key = at / NP;
      int piece = (at - key * NP) ^ (key & 7);
      if (NP > WS * 4 && piece >= WS * 4) piece = 0;          // (room that no fragment reads)
      const uintptr_t from = (unsigned)__shfl(low, key, ZA_WAVE) | (uintptr_t)(unsigned)__shfl(high, key, ZA_WAVE) << 32;
      lds_request((const bf16_t*)from + piece * 8, to + i * 1024);
    }
  };
  request(range_lo);

  const int pos_q = row_ok ? positions[tok] : -1;
  bf16x8_t qf[WS];
  {
    const bf16_t* qrow = q + ((size_t)tok * H + h) * W + kq * 8;      // (a row that is not there: masked)
#pragma unroll
    for (int ks = 0; ks < WS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8_t*>(qrow + ks * 32);
  }
  float m = -INFINITY, l = 0.f;
  f32x4_t o[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int k_at = (wave * 16 + r16) * NP * 16 + ((kq ^ (r16 & 7)) << 4);
  const int v_key = kq * 8 + (r16 >> 2);                      // of the first four of a lane group's eight keys

  for (int tile0 = range_lo; tile0 <= range_hi; tile0 += LD_KT) {
    __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
    __syncthreads();
    // ---- scores: fragments four ahead of their products, which go to two accumulators
    f32x4_t s = {0.f, 0.f, 0.f, 0.f}, u = s;
    bf16x8_t kf[2][4];
    auto read_keys = [&](int g, bf16x8_t (&f)[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (g * 4 + i < WS)
          f[i] = *reinterpret_cast<const bf16x8_t*>(Ks + (k_at ^ (((g * 4 + i) & 1) << 6)) + (g * 4 + i) / 2 * 128);
    };
    read_keys(0, kf[0]);
#pragma unroll
    for (int g = 0; g < (WS + 3) / 4; ++g) {
      if (g * 4 + 4 < WS) read_keys(g + 1, kf[(g + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ks = g * 4 + i;
        if (ks >= WS) continue;
        if (ks & 1) u = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[g & 1][i], qf[ks], u, 0, 0, 0);
        else s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[g & 1][i], qf[ks], s, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    s += u;
    const int kp0 = tile0 + wave * 16 + kq * 4, last = min(pos_q, range_hi);
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = kp0 + i <= last ? s[i] * scale_log2 : -INFINITY;
      top = fmaxf(top, s[i]);
    }
    top = fmaxf(top, __shfl_xor(top, 16, ZA_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, ZA_WAVE));
    if (kq == 0) Xs[r16 * LD_NW + wave] = top;
    __syncthreads();
    float m_new = m;
#pragma unroll
    for (int w = 0; w < LD_NW; w += 4) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(&Xs[r16 * LD_NW + w]);
      m_new = fmaxf(m_new, fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
    }
    const float m_use = m_new > -INFINITY ? m_new : 0.f;
    const float alpha = m == m_new ? 1.0f : exp2f(m - m_use);
    m = m_new;
    bf16x4_t p, rest;
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float e = exp2f(s[i] - m_use);
      p[i] = (bf16_t)e;
      rest[i] = (bf16_t)(e - (float)p[i]);
      psum += (float)p[i] + (float)rest[i];
    }
    l = l * alpha + psum;
    // (weights of a row in pieces of eight keys, piece ^ (row % 8))
    const int p_at = r16 * (LD_KT * 2) + (((wave * 2 + (kq >> 1)) ^ (r16 & 7)) << 4) + (kq & 1) * 8;
    *reinterpret_cast<bf16x4_t*>(Ps + p_at) = p;
    *reinterpret_cast<bf16x4_t*>(Rs + p_at) = rest;
    __syncthreads();
    // ---- values
    auto values = [&](auto whole) {      // (of blocks of 32 keys, those in the range)
#pragma unroll
      for (int t = 0; t < OT; ++t) o[t] *= alpha;
#pragma unroll
      for (int kk = 0; kk < LD_KT / 32; ++kk) {
        if (!decltype(whole)::value && tile0 + kk * 32 > range_hi) continue;
        const int at = r16 * (LD_KT * 2) + (((kk * 4 + kq) ^ (r16 & 7)) << 4);
        const bf16x8_t pf = *reinterpret_cast<const bf16x8_t*>(Ps + at), rf = *reinterpret_cast<const bf16x8_t*>(Rs + at);
        bf16x8_t vf[OT];
#pragma unroll
        for (int t = 0; t < OT; ++t) {
          bf16x4_t half[2];
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            const int key = kk * 32 + v_key + hf * 4, piece = (wave * OT + t) * 2 + ((r16 >> 1) & 1);
            half[hf] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)(
                Ks + key * NP * 16 + ((piece ^ (key & 7)) << 4) + (r16 & 1) * 8));
          }
          vf[t] = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
        for (int t = 0; t < OT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], rf, o[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < OT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], pf, o[t], 0, 0, 0);
      }
    };
    if (tile0 + LD_KT - 32 <= range_hi) values(std::true_type{});
    else values(std::false_type{});
    if (tile0 + LD_KT <= range_hi) {
      __syncthreads();                                        // the tile has been read
      request(tile0 + LD_KT);
    }
  }

  // the rows' sums meet like their maxima
  l += __shfl_xor(l, 16, ZA_WAVE);
  l += __shfl_xor(l, 32, ZA_WAVE);
  __syncthreads();
  if (kq == 0) Xs[r16 * LD_NW + wave] = l;
  __syncthreads();
  if (!row_ok) return;
  float lt = 0.f;
#pragma unroll
  for (int w = 0; w < LD_NW; ++w) lt += Xs[r16 * LD_NW + w];
  if (nsplit == 1) {
    if (sink) lt += exp2f(sink[h] * LM_LOG2E - m);
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    bf16_t* orow = out + ((size_t)tok * H + h) * R + wave * OT * 16 + kq * 4;
#pragma unroll
    for (int t = 0; t < OT; ++t) {
      bf16x4_t v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(o[t][i] * inv);
      *reinterpret_cast<bf16x4_t*>(orow + t * 16) = v;
    }
  } else {
    const size_t pidx = ((size_t)tok * H + h) * nsplit + z;
    float* pa = part_acc + pidx * R + wave * OT * 16 + kq * 4;
#pragma unroll
    for (int t = 0; t < OT; ++t) *reinterpret_cast<f32x4_t*>(pa + t * 16) = o[t];
    if (wave == 0 && kq == 0) {
      part_ml[pidx * 2] = m * LM_LN2;
      part_ml[pidx * 2 + 1] = lt;
    }
  }
}

// The partial results of a row's ranges -> the row.  `base2`: the partial maxima are whole
// numbers on the base-2 scale (what the matrix-core kernel keeps), so a partial result's
// weight 2^(m_z - m) is an exact power of two.
template <typename T>
__global__ void __launch_bounds__(64)
latent_combine_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                      T* __restrict__ out, int R, int nsplit, int base2,
                      const float* __restrict__ sink, int H) {
  const size_t row = blockIdx.x;  // token * H + head
  const int lane = threadIdx.x;
  float mx = -INFINITY;
  for (int z = 0; z < nsplit; ++z) mx = fmaxf(mx, part_ml[(row * nsplit + z) * 2]);
  float total = 0.f;
  float acc[LA_RPL];
#pragma unroll
  for (int c = 0; c < LA_RPL; ++c) acc[c] = 0.f;
  for (int z = 0; z < nsplit; ++z) {
    const float mz = part_ml[(row * nsplit + z) * 2];
    const float lz = part_ml[(row * nsplit + z) * 2 + 1];
    if (!(mz > -INFINITY)) continue;
    const float w = base2 ? ldexpf(1.0f, (int)(mz - mx)) : expf(mz - mx);
    total += lz * w;
    const float* pa = part_acc + (row * nsplit + z) * R;
#pragma unroll
    for (int c = 0; c < LA_RPL; ++c) {
      const int dd = lane + 64 * c;
      if (dd < R) acc[c] = fmaf(pa[dd], w, acc[c]);
    }
  }
  if (sink && mx > -INFINITY) {
    const float sk = sink[row % H];
    total += base2 ? exp2f(sk * 1.4426950408889634f - mx) : expf(sk - mx);
  }
  const float inv = total > 0.f ? 1.0f / total : 0.f;
#pragma unroll
  for (int c = 0; c < LA_RPL; ++c) {
    const int dd = lane + 64 * c;
    if (dd < R) out[row * R + dd] = from_f32<T>(acc[c] * inv);
  }
}

template <typename T, int KT>
static int launch_latent_attention(const void* q, void* out, const void* plane,
                                   long long page_stride, const int* block_table, int bt_stride,
                                   const int* positions, const int* wi_seq, const int* wi_row0,
                                   const int* wi_count, int n_items, float* part_acc,
                                   float* part_ml, int H, int HC, int W, int R, int page_size,
                                   float scale, int keys_per_split, int nsplit, const float* sink,
                                   hipStream_t stream) {
  const size_t shmem = ((size_t)KT * (W + 1) + (size_t)LA_MAX_ROWS * W + LA_WAVES * 64) * sizeof(float);
  auto kernel = latent_attention_kernel<T, KT>;
  static size_t allowed = 0;
  if (shmem > allowed) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e != hipSuccess) return (int)e;
    allowed = shmem;
  }
  dim3 grid(n_items, (H + HC - 1) / HC, nsplit), block(256);
  hipLaunchKernelGGL(kernel, grid, block, shmem, stream, (const T*)q, (T*)out, (const T*)plane,
                     page_stride, block_table, bt_stride, positions, wi_seq, wi_row0, wi_count,
                     part_acc, part_ml, H, HC, W, R, page_size, scale, keys_per_split, nsplit, sink);
  return za_launch_status();
}

// The same for up to 64 ranges, a workgroup a row: the first wave turns the ranges' maxima
// and sums into weights, then every thread adds up its elements over the ranges, in the
// order of the ranges, with loads that do not wait for each other.
template <typename T>
__global__ void __launch_bounds__(256)
latent_combine_wide_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                           T* __restrict__ out, int R, int nsplit, const float* __restrict__ sink,
                           int H) {
  __shared__ float wz[64];
  __shared__ float tot;
  __shared__ int used;            // ranges up to the last that has a result (a sum of -1: it has none)
  const size_t row = blockIdx.x;  // token * H + head
  const int tid = threadIdx.x;
  if (tid < 64) {
    float mz = -INFINITY, lz = -1.f;
    if (tid < nsplit) {
      mz = part_ml[(row * nsplit + tid) * 2];
      lz = part_ml[(row * nsplit + tid) * 2 + 1];
    }
    const unsigned long long there = __ballot(lz != -1.f);
    if (lz == -1.f) lz = 0.f;
    if (tid == 0) used = there ? 64 - __clzll((long long)there) : 0;
    const float mx = wave_max(mz);
    const float w = mz > -INFINITY ? expf(mz - mx) : 0.f;
    float total = wave_sum(lz * w);
    if (sink && mx > -INFINITY) total += expf(sink[row % H] - mx);
    wz[tid] = w;
    if (tid == 0) tot = total;
  }
  __syncthreads();
  const float inv = tot > 0.f ? 1.0f / tot : 0.f;
  for (int dd = tid; dd < R; dd += 256) {
    const float* pa = part_acc + row * nsplit * R + dd;
    float acc = 0.f;
#pragma unroll 4
    for (int z = 0; z < used; ++z) acc = fmaf(pa[(size_t)z * R], wz[z], acc);
    out[row * R + dd] = from_f32<T>(acc * inv);
  }
}

template <int WS, int RT, bool DECODE>
static int launch_latent_mfma(const void* q, void* out, const void* plane, long long page_stride,
                              const int* block_table, int bt_stride, const int* positions,
                              const int* wi_seq, const int* wi_row0, const int* wi_count,
                              int n_items, float* part_acc, float* part_ml, int H, int W, int R,
                              int page_size, float scale, int keys_per_split, int nsplit,
                              const float* sink, hipStream_t stream) {
  const int ws = (W + 31) / 32, rt = (R + 15) / 16;
  const size_t shmem = ((size_t)LM_KT * (ws * 32 + 8) + (size_t)8 * lm_vp(rt) * LM_VS) * sizeof(bf16_t) +
                       (DECODE ? 4 * 64 * 8 * sizeof(float) : 0);
  auto kernel = DECODE ? latent_decode_mfma_kernel<WS, RT> : latent_attention_mfma_kernel<WS, RT>;
  static size_t allowed = 0;
  if (shmem > allowed) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e != hipSuccess) return (int)e;
    allowed = shmem;
  }
  int shift = -1;
  if ((page_size & (page_size - 1)) == 0) {
    shift = 0;
    while ((1 << shift) < page_size) ++shift;
  }
  const int most = DECODE ? 16 : 64;
  const int HC = H < most ? H : most;
  dim3 grid(n_items, (H + HC - 1) / HC, nsplit), block(LM_NT);
  hipLaunchKernelGGL(kernel, grid, block, shmem, stream, (const bf16_t*)q, (bf16_t*)out,
                     (const bf16_t*)plane, page_stride, block_table, bt_stride, positions, wi_seq,
                     wi_row0, wi_count, part_acc, part_ml, H, HC, W, R, page_size, shift,
                     scale * LM_LOG2E, keys_per_split, nsplit, sink);
  return za_launch_status();
}

template <int RT, int DT>
static int launch_latent_prefill(const void* q, void* out, const void* plane, long long page_stride,
                                 const int* block_table, int bt_stride, const int* positions,
                                 const int* wi_seq, const int* wi_row0, const int* wi_count,
                                 int n_items, float* part_acc, float* part_ml, int H, int W, int R,
                                 int page_size, float scale, int keys_per_split, int nsplit,
                                 const float* sink, hipStream_t stream) {
  using S = LpShape<RT, DT>;
  auto kernel = latent_prefill_mfma_kernel<RT, DT>;
  static bool allowed = false;
  if (!allowed) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  int shift = 0;
  while ((1 << shift) < page_size) ++shift;
  const int HC = H < 64 ? H : 64;
  dim3 grid(n_items, (H + HC - 1) / HC, nsplit), block(LP_NT);
  hipLaunchKernelGGL(kernel, grid, block, S::LDS, stream, (const bf16_t*)q, (bf16_t*)out,
                     (const bf16_t*)plane, page_stride, block_table, bt_stride, positions, wi_seq,
                     wi_row0, wi_count, part_acc, part_ml, H, HC, shift,
                     scale * LM_LOG2E, keys_per_split, nsplit, sink);
  return za_launch_status();
}

template <int RT, int DT>
static int launch_latent_range(const void* q, void* out, const void* plane, long long page_stride,
                               const int* block_table, int bt_stride, const int* positions, const int* wi_seq,
                               const int* wi_row0, const int* wi_count, int n_items, float* part_acc, float* part_ml,
                               int H, int W, int R, int page_size, float scale, int keys_per_split, int nsplit,
                               const float* sink, hipStream_t stream) {
  auto kernel = latent_decode_range_kernel<RT, DT>;
  constexpr size_t LDS = LdShape<RT, DT>::LDS;
  static bool allowed = false;
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  int shift = 0;
  while ((1 << shift) < page_size) ++shift;
  const int HC = H < 16 ? H : 16;
  hipLaunchKernelGGL(kernel, dim3(n_items, (H + HC - 1) / HC, nsplit), dim3(LD_NW * 64), LDS, stream, (const bf16_t*)q,
                     (bf16_t*)out, (const bf16_t*)plane, page_stride, block_table, bt_stride, positions, wi_seq, wi_row0,
                     wi_count, part_acc, part_ml, H, HC, shift, scale * LM_LOG2E, keys_per_split, nsplit, sink);
  return za_launch_status();
}

// The matrix-core form: bfloat16, `width` and `kv_rank` multiples of 8.  `waves`: 4 (work
// items of at most 64 / min(heads, 64) tokens, 16 rows a wave) or 1 (single tokens, as a
// step that only decodes has: heads in chunks of 16 whose rows the four waves share).
// Arguments otherwise as za_latent_attention.
extern "C" int za_latent_attention_mfma(const void* q, void* out, const void* plane,
                                        long long page_stride, const int* block_table,
                                        int bt_stride, const int* positions, const int* wi_seq,
                                        const int* wi_row0, const int* wi_count, int n_items,
                                        int n_tokens, float* part_acc, float* part_ml, int heads,
                                        int width, int kv_rank, int page_size, float scale,
                                        int keys_per_split, int nsplit, const float* sink,
                                        int waves, hipStream_t stream) {
  if (n_items == 0 || n_tokens == 0) return 0;
  if (n_items < 0 || heads <= 0 || width <= 0 || kv_rank <= 0 || kv_rank > width ||
      page_size <= 0 || bt_stride <= 0 || nsplit < 1 || !q || !out || !plane || !block_table ||
      !positions || !wi_seq || !wi_row0 || !wi_count ||
      page_stride < (long long)page_size * width || (waves != 1 && waves != 4))
    return ZA_ERR_ARG;
  if (width % 8 || kv_rank % 8 || width > LA_MAX_W || kv_rank > LA_MAX_R || nsplit > 65535)
    return ZA_ERR_UNSUPPORTED;
  if (nsplit > 1 && (!part_acc || !part_ml || keys_per_split <= 0 || keys_per_split % 64 != 0))
    return ZA_ERR_ARG;
  const int ws = (width + 31) / 32, rt = (kv_rank + 15) / 16;
  int rc;
#define ZA_LM_ARGS                                                                              \
  q, out, plane, page_stride, block_table, bt_stride, positions, wi_seq, wi_row0, wi_count,     \
      n_items, part_acc, part_ml, heads, width, kv_rank, page_size, scale, keys_per_split,      \
      nsplit, sink, stream
  const int rotated = width - kv_rank;
  const bool whole = (kv_rank == 128 || kv_rank == 256 || kv_rank == 512) && rotated % 32 == 0 && rotated <= 64 &&
                     (page_size & (page_size - 1)) == 0;
#define ZA_LP(RT)                                                                               \
  rc = rotated == 0    ? launch_latent_prefill<RT, 0>(ZA_LM_ARGS)                               \
       : rotated == 32 ? launch_latent_prefill<RT, 1>(ZA_LM_ARGS)                               \
                       : launch_latent_prefill<RT, 2>(ZA_LM_ARGS)
#define ZA_LD(RT)                                                                               \
  rc = rotated == 0    ? launch_latent_range<RT, 0>(ZA_LM_ARGS)                                 \
       : rotated == 32 ? launch_latent_range<RT, 1>(ZA_LM_ARGS)                                 \
                       : launch_latent_range<RT, 2>(ZA_LM_ARGS)
  if (waves == 1 && whole) {
    if (kv_rank == 128) ZA_LD(8);
    else if (kv_rank == 256) ZA_LD(16);
    else ZA_LD(32);
  } else if (waves == 4 && whole) {
    if (kv_rank == 128) ZA_LP(8);
    else if (kv_rank == 256) ZA_LP(16);
    else ZA_LP(32);
  } else if (ws <= 6 && rt <= 8)
    rc = waves == 4 ? launch_latent_mfma<6, 8, false>(ZA_LM_ARGS)
                    : launch_latent_mfma<6, 8, true>(ZA_LM_ARGS);
  else if (ws <= 10 && rt <= 16)
    rc = waves == 4 ? launch_latent_mfma<10, 16, false>(ZA_LM_ARGS)
                    : launch_latent_mfma<10, 16, true>(ZA_LM_ARGS);
  else
    rc = waves == 4 ? launch_latent_mfma<18, 32, false>(ZA_LM_ARGS)
                    : launch_latent_mfma<18, 32, true>(ZA_LM_ARGS);
#undef ZA_LP
#undef ZA_LD
#undef ZA_LM_ARGS
  if (rc != 0 || nsplit == 1) return rc;
  dim3 grid((unsigned)((size_t)n_tokens * heads));
  if (nsplit <= 64)
    hipLaunchKernelGGL((latent_combine_wide_kernel<bf16_t>), grid, dim3(256), 0, stream, part_acc,
                       part_ml, (bf16_t*)out, kv_rank, nsplit, sink, heads);
  else
    hipLaunchKernelGGL((latent_combine_kernel<bf16_t>), grid, dim3(64), 0, stream, part_acc,
                       part_ml, (bf16_t*)out, kv_rank, nsplit, 0, sink, heads);
  return za_launch_status();
}

// q: [T][H][W] folded queries; out: [T][H][R]; plane: the cache, a page's rows one after
// the other, `page_stride` elements from page to page.  Work items: (request, first row,
// rows), each with at most LA_MAX_ROWS / min(H, LA_MAX_ROWS) rows.
extern "C" int za_latent_attention(const void* q, void* out, const void* plane,
                                   long long page_stride, const int* block_table, int bt_stride,
                                   const int* positions, const int* wi_seq, const int* wi_row0,
                                   const int* wi_count, int n_items, int n_tokens, float* part_acc,
                                   float* part_ml, int dtype, int heads, int width, int kv_rank,
                                   int page_size, float scale, int keys_per_split, int nsplit,
                                   const float* sink, hipStream_t stream) {
  if (n_items == 0 || n_tokens == 0) return 0;
  if (n_items < 0 || heads <= 0 || width <= 0 || kv_rank <= 0 || kv_rank > width ||
      page_size <= 0 || bt_stride <= 0 || nsplit < 1 || !q || !out || !plane || !block_table ||
      !positions || !wi_seq || !wi_row0 || !wi_count ||
      page_stride < (long long)page_size * width)
    return ZA_ERR_ARG;
  if (width > LA_MAX_W || kv_rank > LA_MAX_R || nsplit > 65535) return ZA_ERR_UNSUPPORTED;
  if (nsplit > 1 && (!part_acc || !part_ml || keys_per_split <= 0 || keys_per_split % 64 != 0))
    return ZA_ERR_ARG;
  const int HC = heads < LA_MAX_ROWS ? heads : LA_MAX_ROWS;
  int rc;
#define ZA_LA_ARGS                                                                             \
  q, out, plane, page_stride, block_table, bt_stride, positions, wi_seq, wi_row0, wi_count,    \
      n_items, part_acc, part_ml, heads, HC, width, kv_rank, page_size, scale, keys_per_split, \
      nsplit, sink, stream
  const bool small = width <= 256;
  if (dtype == 0)
    rc = small ? launch_latent_attention<float, 64>(ZA_LA_ARGS)
               : launch_latent_attention<float, 32>(ZA_LA_ARGS);
  else if (dtype == 1)
    rc = small ? launch_latent_attention<bf16_t, 64>(ZA_LA_ARGS)
               : launch_latent_attention<bf16_t, 32>(ZA_LA_ARGS);
  else
    return ZA_ERR_UNSUPPORTED;
#undef ZA_LA_ARGS
  if (rc != 0 || nsplit == 1) return rc;
  dim3 grid((unsigned)((size_t)n_tokens * heads)), block(64);
  if (dtype == 0)
    hipLaunchKernelGGL((latent_combine_kernel<float>), grid, block, 0, stream, part_acc, part_ml,
                       (float*)out, kv_rank, nsplit, 0, sink, heads);
  else
    hipLaunchKernelGGL((latent_combine_kernel<bf16_t>), grid, block, 0, stream, part_acc, part_ml,
                       (bf16_t*)out, kv_rank, nsplit, 0, sink, heads);
  return za_launch_status();
}
