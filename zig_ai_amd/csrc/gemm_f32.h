// 32-bit products on the matrix cores' 32-bit instruction (v_mfma_f32_16x16x4_f32: every
// product and sum in 32-bit, as FMA has them).
//
// The order of an element's sum is the same in every kernel here, whatever tile or workgroup
// it falls in and however many rows the product has, so that a token's result does not depend
// on what else is in its step.  K is cut into chains of F32_CHAIN elements.  A chain starts at
// zero and takes sixteen elements of k at a time with four instructions, instruction j those at
// 4 g + j for lane group g = 0 .. 3 (a lane then reads four consecutive elements); the chains'
// sums are added up in their order.  Elements of K beyond the operand count as zeros.
//
// Lane l of 16x16x4: supplies row l % 16 and k element l / 16 of either operand, receives rows
// (l / 16) * 4 .. + 3 of the first operand's sixteen and column l % 16 of the second's.  The
// weights are the first operand: a lane ends with four consecutive outputs of one row.
#pragma once

#include "common.h"

#define F32_CHAIN 128

// Four consecutive elements of a row at k, zeros beyond K.  VEC: K is a multiple of four and
// the operand lies on 16 bytes (8 for bfloat16), so four elements are inside together.
template <typename T, bool VEC>
__device__ __forceinline__ f32x4_t f32_load4(const T* __restrict__ row, int k, int K) {
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    if (k < K) {
      if constexpr (sizeof(T) == 4) {
        v = *reinterpret_cast<const f32x4_t*>(row + k);
      } else {
        const bf16x4_t b = *reinterpret_cast<const bf16x4_t*>(row + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (float)b[i];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k + i < K) v[i] = to_f32<T>(row[k + i]);
  }
  return v;
}

template <typename TC>
__device__ __forceinline__ void f32_store4(TC* __restrict__ C, const float* __restrict__ bias, f32x4_t v, int m,
                                           int n, int N, bool wide) {
  TC* at = C + (size_t)m * N + n;
  if (bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) v[r] += bias[n + r];
  }
  if (sizeof(TC) == 4 && wide) {
    if (n < N) *reinterpret_cast<f32x4_t*>(at) = v;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) at[r] = from_f32<TC>(v[r]);
  }
}

// Many rows: KG groups of four waves (2 x 2) take BM rows and BN outputs, each group every KG-th
// chain of K, 32 elements of k at a time through two places in LDS of its own, the next ones on
// their way from memory meanwhile; at a chain's end the groups' sums meet in LDS, where the first
// group adds them in their order.  A row of 36 floats lets the sixteen rows that a quarter of a
// wave reads fall into different banks.
#define F32_BK 32
#define F32_LD (F32_BK + 4)

// `a_at(r)` and `w_at(r)` name the rows of the tile (some readable row where there is none),
// `store(r, n, v)` takes the sums of row r: v[j] are those of outputs n + 16 j .. + 3.
template <typename TA, int BM, int BN, int KG, bool VEC, typename AAt, typename WAt, typename Store>
__device__ __forceinline__ void f32_tile(int K, AAt a_at, WAt w_at, Store store) {
  constexpr int TM = BM / 32, TN = BN / 32, LA = BM / 32, LW = BN / 32, STEPS = F32_CHAIN / F32_BK;
  __shared__ __attribute__((aligned(16))) float As[KG][2][BM * F32_LD];
  __shared__ __attribute__((aligned(16))) float Ws[KG][2][BN * F32_LD];
  __shared__ f32x4_t sums[KG > 1 ? KG - 1 : 1][KG > 1 ? TM * TN * 256 : 1];
  const int group = threadIdx.x >> 8;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lrow = tid >> 3, lk = (tid & 7) * 4;
  const TA* a_row[LA];
  const float* w_row[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) a_row[i] = a_at(lrow + 32 * i);
#pragma unroll
  for (int i = 0; i < LW; ++i) w_row[i] = w_at(lrow + 32 * i);
  f32x4_t ra[LA], rw[LW];
  // step s of the group: a chain's steps, then those of the chain KG on
  auto k_of = [&](int s) { return ((s / STEPS) * KG + group) * F32_CHAIN + (s % STEPS) * F32_BK; };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < LA; ++i)
      ra[i] = f32_load4<TA, VEC>(a_row[i], k0 + lk, K);
#pragma unroll
    for (int i = 0; i < LW; ++i)
      rw[i] = f32_load4<float, VEC>(w_row[i], k0 + lk, K);
  };
  auto stash = [&](int p) {
#pragma unroll
    for (int i = 0; i < LA; ++i)
      *reinterpret_cast<f32x4_t*>(&As[group][p][(lrow + 32 * i) * F32_LD + lk]) = ra[i];
#pragma unroll
    for (int i = 0; i < LW; ++i)
      *reinterpret_cast<f32x4_t*>(&Ws[group][p][(lrow + 32 * i) * F32_LD + lk]) = rw[i];
  };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = zero;
  const int frow = lane & 15, fk = (lane >> 4) * 4;
  // all groups walk the same number of steps (beyond K they take zeros, which add nothing)
  const int steps = K <= KG * F32_CHAIN ? (min(K, F32_CHAIN) + F32_BK - 1) / F32_BK
                                        : (K + KG * F32_CHAIN - 1) / (KG * F32_CHAIN) * STEPS;
  fetch(k_of(0));
  stash(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int p = s & 1;
    const bool more = s + 1 < steps;
    if (more) fetch(k_of(s + 1));
#pragma unroll
    for (int ks = 0; ks < F32_BK; ks += 16) {
      f32x4_t fa[TM], fw[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[i] = *reinterpret_cast<const f32x4_t*>(&As[group][p][(wm + i * 16 + frow) * F32_LD + ks + fk]);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fw[j] = *reinterpret_cast<const f32x4_t*>(&Ws[group][p][(wn + j * 16 + frow) * F32_LD + ks + fk]);
      // (one element of k for all tiles, then the next: an accumulator's own products are
      // TM * TN instructions apart)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[j][e], fa[i][e], acc[i][j], 0, 0, 0);
    }
    if (more) stash(p ^ 1);
    const bool chain_ends = !more || (s + 1) % STEPS == 0;
    if (KG > 1 && chain_ends && group > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sums[group - 1][(i * TN + j) * 256 + tid] = acc[i][j];
          acc[i][j] = zero;
        }
    }
    __syncthreads();
    if (chain_ends && group == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = zero;
#pragma unroll
          for (int g = 1; g < KG; ++g) total[i][j] += sums[g - 1][(i * TN + j) * 256 + tid];
        }
    }
  }
  if (group > 0) return;
#pragma unroll
  for (int i = 0; i < TM; ++i) store(wm + i * 16 + frow, wn + fk, total[i]);
}

// The same tile, groups and order of sums for 32-bit rows on 16 bytes and K in whole steps of 32: the
// steps go from memory into NS places of LDS without passing registers, NS - 1 of them under way (the
// tile above has one, in registers, and waits for memory where the weights come from there).  A row's
// eight pieces of four elements lie in the order piece ^ (row % 8), so that the sixteen rows that a
// fragment is read from fall into different banks.  Reads of LDS and their wait stand in one block: the
// compiler would have each wait for every request under way to LDS.
template <int BM, int BN, int KG, int NS, typename AAt, typename WAt, typename Store>
__device__ __forceinline__ void f32_tile_async(int K, AAt a_at, WAt w_at, Store store) {
  constexpr int TM = BM / 32, TN = BN / 32, LA = BM / 32, LW = BN / 32, STEPS = F32_CHAIN / F32_BK;
  static_assert((TM == 2 && TN == 2) || (TM == 1 && TN == 2) || (TM == 1 && TN == 1), "see take");
  __shared__ __attribute__((aligned(16))) float As[KG][NS][BM * F32_BK];
  __shared__ __attribute__((aligned(16))) float Ws[KG][NS][BN * F32_BK];
  __shared__ __attribute__((aligned(16))) f32x4_t sums[KG > 1 ? KG - 1 : 1][KG > 1 ? TM * TN * 256 : 1];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lrow = wave * 8 + (lane >> 3), piece = ((lane & 7) ^ (lane >> 3)) * 4;
  const float *a_row[LA], *w_row[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) a_row[i] = a_at(lrow + 32 * i) + piece;
#pragma unroll
  for (int i = 0; i < LW; ++i) w_row[i] = w_at(lrow + 32 * i) + piece;
  // step s of the group: a chain's steps, then those of the chain KG on
  auto k_of = [&](int s) { return ((s / STEPS) * KG + group) * F32_CHAIN + (s % STEPS) * F32_BK; };
  auto request = [&](int s, int p) {
    const int k0 = k_of(s) < K ? k_of(s) : 0;      // (a step beyond K: not multiplied)
#pragma unroll
    for (int i = 0; i < LA; ++i) lds_request(a_row[i] + k0, &As[group][p][(32 * i + wave * 8) * F32_BK]);
#pragma unroll
    for (int i = 0; i < LW; ++i) lds_request(w_row[i] + k0, &Ws[group][p][(32 * i + wave * 8) * F32_BK]);
  };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = zero;
  const int frow = lane & 15, fk = lane >> 4;
  const unsigned slot[2] = {(unsigned)((fk ^ (frow & 7)) * 16), (unsigned)(((4 + fk) ^ (frow & 7)) * 16)};
  f32x4_t fa[2][TM], fw[2][TN];
  auto take = [&](int p) {
    const unsigned w = lds_address(&Ws[group][p][(wn + frow) * F32_BK]), a = lds_address(&As[group][p][(wm + frow) * F32_BK]);
    const unsigned w0 = w + slot[0], w1 = w + slot[1], a0 = a + slot[0], a1 = a + slot[1];
    if constexpr (TM == 2) {
      asm volatile(
          "ds_read_b128 %0, %8 offset:0\n" "ds_read_b128 %1, %8 offset:2048\n"
          "ds_read_b128 %2, %10 offset:0\n" "ds_read_b128 %3, %10 offset:2048\n"
          "ds_read_b128 %4, %9 offset:0\n" "ds_read_b128 %5, %9 offset:2048\n"
          "ds_read_b128 %6, %11 offset:0\n" "ds_read_b128 %7, %11 offset:2048\n"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(fw[0][0]), "=&v"(fw[0][1]), "=&v"(fa[0][0]), "=&v"(fa[0][1]),
            "=&v"(fw[1][0]), "=&v"(fw[1][1]), "=&v"(fa[1][0]), "=&v"(fa[1][1])
          : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
          : "memory");
    } else if constexpr (TN == 2) {
      asm volatile(
          "ds_read_b128 %0, %6 offset:0\n" "ds_read_b128 %1, %6 offset:2048\n"
          "ds_read_b128 %2, %8 offset:0\n" "ds_read_b128 %3, %7 offset:0\n"
          "ds_read_b128 %4, %7 offset:2048\n" "ds_read_b128 %5, %9 offset:0\n"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(fw[0][0]), "=&v"(fw[0][1]), "=&v"(fa[0][0]), "=&v"(fw[1][0]),
            "=&v"(fw[1][1]), "=&v"(fa[1][0])
          : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
          : "memory");
    } else {
      asm volatile(
          "ds_read_b128 %0, %4 offset:0\n" "ds_read_b128 %1, %6 offset:0\n"
          "ds_read_b128 %2, %5 offset:0\n" "ds_read_b128 %3, %7 offset:0\n"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(fw[0][0]), "=&v"(fa[0][0]), "=&v"(fw[1][0]), "=&v"(fa[1][0])
          : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
          : "memory");
    }
  };
  // the other groups' sums of the chain that has ended, behind a barrier
  auto add_sums = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 1; g < KG; ++g) {
          f32x4_t v;
          asm volatile("ds_read_b128 %0, %1\ns_waitcnt lgkmcnt(0)"
                       : "=&v"(v) : "v"(lds_address(&sums[g - 1][(i * TN + j) * 256 + tid])) : "memory");
          total[i][j] += v;
        }
  };
  // all groups walk the same number of steps
  const int steps = K <= KG * F32_CHAIN ? (min(K, F32_CHAIN) + F32_BK - 1) / F32_BK
                                        : (K + KG * F32_CHAIN - 1) / (KG * F32_CHAIN) * STEPS;
#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    if (i < steps) request(i, i);
  int p = 0, q = NS - 1;
  bool pending = false;
  for (int s = 0; s < steps; ++s) {
    // this step's tiles have arrived when only those requested after them are on their way
    if (s + NS - 2 < steps) __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 2) * (LA + LW)));
    else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
    __builtin_amdgcn_s_barrier();
    take(p);
    if (s + NS - 1 < steps) request(s + NS - 1, q);
    if (KG > 1 && pending && group == 0) add_sums();
    pending = false;
    if (k_of(s) < K) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[h][j][e], fa[h][i][e], acc[i][j], 0, 0, 0);
    }
    if (s + 1 == steps || (s + 1) % STEPS == 0) {
      if (KG == 1 || group == 0) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) total[i][j] += acc[i][j];
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            asm volatile("ds_write_b128 %0, %1" :: "v"(lds_address(&sums[group - 1][(i * TN + j) * 256 + tid])),
                         "v"(acc[i][j]) : "memory");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = zero;
      pending = true;
    }
    __builtin_amdgcn_sched_barrier(0);     // (or the products move behind the next wait)
    p = p + 1 == NS ? 0 : p + 1;
    q = q + 1 == NS ? 0 : q + 1;
  }
  if constexpr (KG > 1) {
    __builtin_amdgcn_s_barrier();
    if (group > 0) return;
    add_sums();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) store(wm + i * 16 + frow, wn + fk * 4, total[i]);
}

template <typename TC, int BM, int BN, int KG, int NS>
__global__ void __launch_bounds__(256 * KG)
gemm_f32_async_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                      TC* __restrict__ C, int M, int N, int K, int m_tiles, int n_tiles, int wide) {
  const int at = blockIdx.x >> 3;                  // (dies and tiles as below)
  const int n_tile = (at / m_tiles) * 8 + (blockIdx.x & 7);
  if (n_tile >= n_tiles) return;
  const int m0 = (at % m_tiles) * BM, n0 = n_tile * BN;
  f32_tile_async<BM, BN, KG, NS>(
      K, [&](int r) { return A + (size_t)min(m0 + r, M - 1) * K; },
      [&](int r) { return W + (size_t)min(n0 + r, N - 1) * K; },
      [&](int r, int n, const f32x4_t(&v)[BN / 32]) {
        if (m0 + r >= M) return;
#pragma unroll
        for (int j = 0; j < BN / 32; ++j) f32_store4<TC>(C, bias, v[j], m0 + r, n0 + n + j * 16, N, wide);
      });
}

template <typename TA, typename TC, int BM, int BN, int KG, bool VEC>
__global__ void __launch_bounds__(256 * KG)
gemm_f32_tile_kernel(const TA* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     TC* __restrict__ C, int M, int N, int K, int m_tiles, int n_tiles, int wide) {
  // workgroups are dealt to the eight dies in turn: the row tiles of one stretch of outputs
  // follow each other on one die, whose cache then holds the weights they share
  const int at = blockIdx.x >> 3;
  const int n_tile = (at / m_tiles) * 8 + (blockIdx.x & 7);
  if (n_tile >= n_tiles) return;
  const int m0 = (at % m_tiles) * BM, n0 = n_tile * BN;
  f32_tile<TA, BM, BN, KG, VEC>(
      K, [&](int r) { return A + (size_t)min(m0 + r, M - 1) * K; },
      [&](int r) { return W + (size_t)min(n0 + r, N - 1) * K; },
      [&](int r, int n, const f32x4_t(&v)[BN / 32]) {
        if (m0 + r >= M) return;
#pragma unroll
        for (int j = 0; j < BN / 32; ++j) f32_store4<TC>(C, bias, v[j], m0 + r, n0 + n + j * 16, N, wide);
      });
}

// Few rows: a workgroup of NW waves takes 16 rows and 16 outputs, and its waves take the
// chains of K in turn, operands straight from memory; NW chains at a time meet in LDS, where
// they are added in their order.
template <typename TA, typename TC, int NW, bool VEC>
__global__ void __launch_bounds__(NW * 64)
gemm_f32_rows_kernel(const TA* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     TC* __restrict__ C, int M, int N, int K, int m_tiles, int n_tiles, int wide) {
  __shared__ f32x4_t sums[2][NW][64];
  const int at = blockIdx.x >> 3;
  const int n_tile = (at / m_tiles) * 8 + (blockIdx.x & 7);
  if (n_tile >= n_tiles) return;
  const int m0 = (at % m_tiles) * 16, n0 = n_tile * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int frow = lane & 15, fk = (lane >> 4) * 4;
  const int chains = (K + F32_CHAIN - 1) / F32_CHAIN;
  const TA* a_row = A + (size_t)min(m0 + frow, M - 1) * K;
  const float* w_row = W + (size_t)min(n0 + frow, N - 1) * K;
  f32x4_t total = {0.f, 0.f, 0.f, 0.f};
  int p = 0;
  for (int c0 = 0; c0 < chains; c0 += NW, p ^= 1) {
    const int c = c0 + wave;
    if (c < chains) {
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
      f32x4_t fa[F32_CHAIN / 16], fw[F32_CHAIN / 16];
#pragma unroll
      for (int b = 0; b < F32_CHAIN / 16; ++b) {
        const int k = c * F32_CHAIN + b * 16 + fk;
        fw[b] = f32_load4<float, VEC>(w_row, k, K);
        fa[b] = f32_load4<TA, VEC>(a_row, k, K);
      }
#pragma unroll
      for (int b = 0; b < F32_CHAIN / 16; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[b][e], fa[b][e], acc, 0, 0, 0);
      sums[p][wave][lane] = acc;
    }
    __syncthreads();
    // (the next round writes the other half, and the one after it behind the next barrier)
    if (wave == 0)
      for (int w = 0; w < NW && c0 + w < chains; ++w) total += sums[p][w][lane];
  }
  if (wave == 0 && m0 + frow < M) f32_store4<TC>(C, bias, total, m0 + frow, n0 + fk, N, wide);
}
