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

#include <type_traits>

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

// The same order of sums for 32-bit rows on 16 bytes and K in whole steps of 32, by four waves without groups: the
// steps go from memory into NS places of LDS without passing registers.  A phase is 16 elements of k, four
// products for each of TM x TN sums, one asm statement: the reads of the next phase's fragments and, in a step's
// second phase, the requests for step s + NS stand between the products, in their shadow, and the wait for the
// reads ends the statement, as their results may only be known to the compiler when they are there.  One
// barrier a step, between its phases: it ends the reads of the step's place and says that the next step has
// arrived.
// Nothing may touch the sums between these statements: another instruction that reads a product's sums has to wait
// some clocks for them, which the compiler does not see to here.  So a chain's steps stand in a row without a
// branch (with one, the compiler copies sums where the ways meet: wrong, and half a step's time), and the last
// whole chain is there once for each number of steps behind it: how many steps are still to be requested and
// are under way at each wait is known where the code is written.  Nor does it see that a chain's first product reads sums that it has just
// cleared, which takes two wait states: the first statement of a chain begins with them.
// 64 x 64 takes 1,150 clocks a step of 1,024 of products, 32 x 64 615 of 512.  A row's eight pieces of four elements
// lie in the order piece ^ (row % 8), so that the sixteen rows that a fragment is read from fall into
// different banks.
#define GF_MF(i, j, e) "v_mfma_f32_16x16x4_f32 %[c" #i #j "], %[w" #j #e "], %[a" #i #e "], %[c" #i #j "]\n"
#define GF_RD(k, p, o) "ds_read_b128 %[n" #k "], %[" #p "] offset:" #o "\n"
// (m0 is set one instruction ahead of the request, which needs that distance)
#define GF_TO(k) "s_mov_b32 m0, %[m" #k "]\n"
#define GF_RQ(k, b) "global_load_lds_dwordx4 %[v" #k "], %[" #b "]\n"
#define GF_FOUR(n, v) [n##0] "v"(v[0]), [n##1] "v"(v[1]), [n##2] "v"(v[2]), [n##3] "v"(v[3])
#define GF_WAIT "s_waitcnt lgkmcnt(0)\n"
#define GF_CLEARED "s_nop 1\n"
#define GF_ALL12(e) GF_MF(0, 0, e) GF_MF(0, 1, e)
#define GF_ALL22(e) GF_ALL12(e) GF_MF(1, 0, e) GF_MF(1, 1, e)
#define GF_START12 GF_MF(0, 0, 0) GF_RD(0, pw, 0) GF_MF(0, 1, 0) GF_RD(1, pw, 2048) GF_RD(2, pa, 0)
#define GF_START22 \
  GF_MF(0, 0, 0) GF_RD(0, pw, 0) GF_MF(0, 1, 0) GF_RD(1, pw, 2048) GF_MF(1, 0, 0) GF_RD(2, pa, 0) GF_MF(1, 1, 0) GF_RD(3, pa, 2048)
#define GF_WITH12                                                                                     \
  GF_MF(0, 0, 1) GF_TO(0) GF_MF(0, 1, 1) GF_RQ(0, bw) GF_MF(0, 0, 2) GF_TO(1) GF_MF(0, 1, 2) GF_RQ(1, bw) \
  GF_MF(0, 0, 3) GF_TO(2) GF_MF(0, 1, 3) GF_RQ(2, ba)
#define GF_WITH22                                                                                         \
  GF_MF(0, 0, 1) GF_TO(0) GF_MF(0, 1, 1) GF_RQ(0, bw) GF_MF(1, 0, 1) GF_TO(1) GF_MF(1, 1, 1) GF_RQ(1, bw)     \
  GF_MF(0, 0, 2) GF_MF(0, 1, 2) GF_TO(2) GF_MF(1, 0, 2) GF_RQ(2, ba) GF_MF(1, 1, 2) GF_TO(3) GF_MF(0, 0, 3) \
  GF_RQ(3, ba) GF_MF(0, 1, 3) GF_MF(1, 0, 3) GF_MF(1, 1, 3)
#define GF_C12 [c00] "+v"(c[0][0]), [c01] "+v"(c[0][1])
#define GF_C22 GF_C12, [c10] "+v"(c[1][0]), [c11] "+v"(c[1][1])
#define GF_N12 [n0] "=&v"(nw[0]), [n1] "=&v"(nw[1]), [n2] "=&v"(na[0])
#define GF_N22 GF_N12, [n3] "=&v"(na[1])
#define GF_IN12 GF_FOUR(w0, w[0]), GF_FOUR(w1, w[1]), GF_FOUR(a0, a[0]), [pw] "v"(pw), [pa] "v"(pa)
#define GF_IN22 GF_IN12, GF_FOUR(a1, a[1])
#define GF_Q12                                                                                              \
  [v0] "v"(q.offw[0]), [m0] "s"(q.tow), [v1] "v"(q.offw[1]), [m1] "s"(q.tow + 4096), [v2] "v"(q.offa[0]),         \
  [m2] "s"(q.toa), [bw] "s"(q.w), [ba] "s"(q.a)
#define GF_Q22 GF_Q12, [v3] "v"(q.offa[1]), [m3] "s"(q.toa + 4096)

struct F32Requests {      // W's and A's offsets of a lane, where its first piece goes, W's and A's base
  const unsigned *offw, *offa;
  unsigned tow, toa;
  const char *w, *a;
};

// FIRST: of a chain, whose sums have just been cleared (then without requests)
template <int TM, int TN, bool REQUEST, bool FIRST>
__device__ __forceinline__ void f32_phase(f32x4_t (&c)[TM][TN], const f32x4_t (&w)[TN], const f32x4_t (&a)[TM],
                                          f32x4_t (&nw)[TN], f32x4_t (&na)[TM], unsigned pw, unsigned pa,
                                          const F32Requests& q) {
  static_assert(TN == 2 && (TM == 2 || TM == 1) && !(REQUEST && FIRST), "one of these");
  if constexpr (TM == 1 && REQUEST)
    asm volatile(GF_START12 GF_WITH12 GF_WAIT : GF_C12, GF_N12 : GF_IN12, GF_Q12 : "memory", "m0");
  else if constexpr (TM == 1 && FIRST)
    asm volatile(GF_CLEARED GF_START12 GF_ALL12(1) GF_ALL12(2) GF_ALL12(3) GF_WAIT : GF_C12, GF_N12 : GF_IN12 : "memory");
  else if constexpr (TM == 1)
    asm volatile(GF_START12 GF_ALL12(1) GF_ALL12(2) GF_ALL12(3) GF_WAIT : GF_C12, GF_N12 : GF_IN12 : "memory");
  else if constexpr (REQUEST)
    asm volatile(GF_START22 GF_WITH22 GF_WAIT : GF_C22, GF_N22 : GF_IN22, GF_Q22 : "memory", "m0");
  else if constexpr (FIRST)
    asm volatile(GF_CLEARED GF_START22 GF_ALL22(1) GF_ALL22(2) GF_ALL22(3) GF_WAIT : GF_C22, GF_N22 : GF_IN22 : "memory");
  else
    asm volatile(GF_START22 GF_ALL22(1) GF_ALL22(2) GF_ALL22(3) GF_WAIT : GF_C22, GF_N22 : GF_IN22 : "memory");
}

// `a_at(r)` and `w_at(r)`: bytes from A and W to the tile's row r (to some readable row where there is none), below
// 4 GB; `store` as above.
template <int BM, int BN, int NS, typename AAt, typename WAt, typename Store>
__device__ __forceinline__ void f32_tile_async(int K, const float* A, const float* W, AAt a_at, WAt w_at, Store store) {
  constexpr int TM = BM / 32, TN = BN / 32, LA = BM / 32, LW = BN / 32, STEPS = F32_CHAIN / F32_BK;
  constexpr int PLACE = (BM + BN) * F32_BK * 4;      // bytes; A's rows behind W's
  __shared__ __attribute__((aligned(16))) char lds[NS * PLACE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lrow = wave * 8 + (lane >> 3), piece = ((lane & 7) ^ (lane >> 3)) * 16;
  unsigned offa[LA], offw[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) offa[i] = a_at(lrow + 32 * i) + piece;
#pragma unroll
  for (int i = 0; i < LW; ++i) offw[i] = w_at(lrow + 32 * i) + piece;
  const int steps = K / F32_BK;
  const unsigned base = lds_address(lds);
  F32Requests q{offw, offa, base + wave * 1024, base + BN * F32_BK * 4 + wave * 1024, (const char*)W, (const char*)A};
  auto behind = [&](bool last) {      // a step's requests, which went to the last place
    const unsigned by = last ? (unsigned)(-(NS - 1) * PLACE) : (unsigned)PLACE;
    q.w += F32_BK * 4;
    q.a += F32_BK * 4;
    q.tow += by;
    q.toa += by;
  };
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (s >= steps) continue;
    auto request = [&](const char* from, unsigned offset, unsigned to) {
      asm volatile("s_mov_b32 m0, %0\n" "s_nop 0\n" "global_load_lds_dwordx4 %1, %2\n"
                   :: "s"(to), "v"(offset), "s"(from) : "memory", "m0");
    };
#pragma unroll
    for (int i = 0; i < LW; ++i) request(q.w, offw[i], q.tow + i * 4096);
#pragma unroll
    for (int i = 0; i < LA; ++i) request(q.a, offa[i], q.toa + i * 4096);
    behind(s == NS - 1);
  }
  f32x4_t total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) total[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int frow = lane & 15, fk = lane >> 4;
  const unsigned half[2] = {(unsigned)((fk ^ (frow & 7)) * 16), (unsigned)(((4 + fk) ^ (frow & 7)) * 16)};
  const unsigned rw = base + (wn + frow) * F32_BK * 4, ra = base + (BN + wm + frow) * F32_BK * 4;
  auto meet = [&]() {      // nothing moves over it
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (steps >= NS) __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 1) * (LA + LW)));
  else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
  meet();
  f32x4_t a0[TM], w0[TN], a1[TM], w1[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    asm volatile("ds_read_b128 %0, %1\n" "s_waitcnt lgkmcnt(0)" : "=&v"(w0[j]) : "v"(rw + half[0] + j * 2048) : "memory");
#pragma unroll
  for (int i = 0; i < TM; ++i)
    asm volatile("ds_read_b128 %0, %1\n" "s_waitcnt lgkmcnt(0)" : "=&v"(a0[i]) : "v"(ra + half[0] + i * 2048) : "memory");
  unsigned at = 0;
  auto chain = [&](auto count, auto behind_it) {      // its steps, and how many (or NS, if more) are behind them
    constexpr int COUNT = decltype(count)::value, BEHIND = decltype(behind_it)::value;
    f32x4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const int follow = COUNT - 1 - u + BEHIND;
      const bool last = at == (NS - 1) * PLACE;
      const unsigned to = last ? 0 : at + PLACE;
      const unsigned pw = rw + at + half[1], pa = ra + at + half[1];
      if (u == 0) f32_phase<TM, TN, false, true>(acc, w0, a0, w1, a1, pw, pa, q);
      else f32_phase<TM, TN, false, false>(acc, w0, a0, w1, a1, pw, pa, q);
      // (the next step has arrived: of what follows it the NS - 2 steps are under way that are left)
      if (follow >= NS - 1) __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 2) * (LA + LW)));
      else if (follow == NS - 2) __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 3) * (LA + LW)));
      else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
      meet();
      // (the last step's reads find an older step's tiles: not used)
      const unsigned qw = rw + to + half[0], qa = ra + to + half[0];
      if (follow >= NS) f32_phase<TM, TN, true, false>(acc, w1, a1, w0, a0, qw, qa, q);
      else f32_phase<TM, TN, false, false>(acc, w1, a1, w0, a0, qw, qa, q);
      behind(last);
      at = to;
    }
    asm volatile("s_nop 15" : "+v"(acc[0][0]));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (i + j > 0) asm volatile("" : "+v"(acc[i][j]));
        total[i][j] += acc[i][j];
      }
  };
  static_assert(NS == 4 && STEPS == 4, "see the waits, and the ends");
  constexpr std::integral_constant<int, 0> none;
  constexpr std::integral_constant<int, 1> one;
  constexpr std::integral_constant<int, 2> two;
  constexpr std::integral_constant<int, 3> three;
  constexpr std::integral_constant<int, 4> four;
  const int whole = steps / STEPS, rest = steps % STEPS;
  for (int c = 1; c < whole; ++c) chain(four, four);
  if (rest == 0) {
    chain(four, none);
  } else if (rest == 1) {
    if (whole > 0) chain(four, one);
    chain(one, none);
  } else if (rest == 2) {
    if (whole > 0) chain(four, two);
    chain(two, none);
  } else {
    if (whole > 0) chain(four, three);
    chain(three, none);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) store(wm + i * 16 + frow, wn + fk * 4, total[i]);
}

template <typename TC, int BM, int BN, int NS>
__global__ void __launch_bounds__(256)
gemm_f32_async_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                      TC* __restrict__ C, int M, int N, int K, int m_tiles, int n_tiles, int wide) {
  const int at = blockIdx.x >> 3;                  // (dies and tiles as below)
  const int n_tile = (at / m_tiles) * 8 + (blockIdx.x & 7);
  if (n_tile >= n_tiles) return;
  const int m0 = (at % m_tiles) * BM, n0 = n_tile * BN;
  // (offsets from the tile's own first rows: operands may hold more than 4 GB)
  f32_tile_async<BM, BN, NS>(
      K, A + (size_t)m0 * K, W + (size_t)n0 * K, [&](int r) { return (unsigned)min(r, M - 1 - m0) * (unsigned)(K * 4); },
      [&](int r) { return (unsigned)min(r, N - 1 - n0) * (unsigned)(K * 4); },
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
