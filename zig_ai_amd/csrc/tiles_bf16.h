// Products of rows with rows, bfloat16 into 32-bit sums on the matrix cores, in tiles of BM rows of
// A x BN rows of W that share K: what the grouped products of experts and the heads' own products
// are made of.
//
// Operand layout of v_mfma_f32_16x16x32_bf16: lane l supplies row (l % 16), k-slots
// (l / 16) * 8 .. + 7 of either operand and receives rows (l / 16) * 4 .. + 3, column
// (l % 16) of the product.
//
// The tiles go through LDS, 64 elements of K a step, from memory into one of NS places in LDS
// without passing registers (global_load_lds, 16 bytes a lane, eight rows of 128 bytes an
// instruction); a row's eight pieces lie in the order piece ^ (row % 8), so that the sixteen rows
// a fragment is read from fall into different banks.  A step waits for its own tiles and the other
// waves, takes its fragments, requests the tiles NS - 1 steps on, into the place the step before it
// has left, and multiplies meanwhile: one barrier a step, NS - 1 steps' tiles under way.  With few
// rows the weights' way from memory bounds it, with many the reads of LDS, which take as long as
// the products (tiles of 64 x 64 a wave).  ONCE: the weights are read past the caches' other contents.  The rows of W are the first operand, so a lane ends with
// four consecutive outputs of one row of A.
#pragma once

#include "common.h"

#define GG_BK 64

// From this many bytes of weights on a product reads them past the caches' other contents: a guess from one product's
// size that its model is larger than the last level's cache (256 MB) holds from one step to the next.
#define ZA_ONCE_BYTES (32LL << 20)

template <int BM, int BN, int NS, bool ONCE = false>
struct TilesBf16 {
  static constexpr int WM = BM >= 64 || BN == 64 ? 2 : 1, WN = 4 / WM;   // waves along the rows of A and of W
  static constexpr int TM = BM / (16 * WM), TN = BN / (16 * WN);
  static_assert((TM == 4 && TN == 4) || (TM == 2 && TN == 4) || (TM == 2 && TN == 2) || (TM == 1 && TN == 2), "see take");
  static constexpr int LA = BM / 32, LW = BN / 32;      // instructions a wave and tile (8 rows each)

  // `arow`, `wrow`: a lane's rows of the tile, 32 i + 8 wave + lane / 8, each at its piece
  // (lane % 8) ^ (lane / 8) of 8 elements (any valid row for those that are not stored); K is a
  // multiple of 8.  acc[i][j][r]: row wm + 16 i + lane % 16 of A and wn + 16 j + lane / 16 * 4 + r
  // of W, with wm = (wave % WM) * (BM / WM) and wn = (wave / WM) * (BN / WN).
  static __device__ __forceinline__ void run(bf16_t (&As)[NS][BM * GG_BK], bf16_t (&Ws)[NS][BN * GG_BK],
                                             int wave, int lane, int K, const bf16_t* const (&arow)[LA],
                                             const bf16_t* const (&wrow)[LW], f32x4_t (&acc)[TM][TN]) {
    const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
    const int piece = (lane & 7) ^ (lane >> 3);
    auto request = [&](int k0, int p) {
#pragma unroll
      for (int i = 0; i < LA; ++i) lds_request(arow[i] + k0, &As[p][(32 * i + wave * 8) * GG_BK]);
#pragma unroll
      for (int i = 0; i < LW; ++i) lds_request<ONCE>(wrow[i] + k0, &Ws[p][(32 * i + wave * 8) * GG_BK]);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int r16 = lane & 15, kq = lane >> 4;
    // The fragments of place p.  (In one block with its own wait: the compiler would have every
    // read of LDS wait for all requests under way to LDS, the next steps' among them.)
    bf16x8_t fa[2][TM], fw[2][TN];
    const unsigned slot[2] = {(unsigned)((kq ^ (r16 & 7)) * 16), (unsigned)(((4 + kq) ^ (r16 & 7)) * 16)};
    auto take = [&](int p) {
      const unsigned w = lds_address(&Ws[p][(wn + r16) * GG_BK]), a = lds_address(&As[p][(wm + r16) * GG_BK]);
      const unsigned w0 = w + slot[0], w1 = w + slot[1], a0 = a + slot[0], a1 = a + slot[1];
      if constexpr (TM == 4 && TN == 4) {
        asm volatile(
            "ds_read_b128 %0, %16 offset:0\n" "ds_read_b128 %1, %16 offset:2048\n"
            "ds_read_b128 %2, %16 offset:4096\n" "ds_read_b128 %3, %16 offset:6144\n"
            "ds_read_b128 %4, %18 offset:0\n" "ds_read_b128 %5, %18 offset:2048\n"
            "ds_read_b128 %6, %18 offset:4096\n" "ds_read_b128 %7, %18 offset:6144\n"
            "ds_read_b128 %8, %17 offset:0\n" "ds_read_b128 %9, %17 offset:2048\n"
            "ds_read_b128 %10, %17 offset:4096\n" "ds_read_b128 %11, %17 offset:6144\n"
            "ds_read_b128 %12, %19 offset:0\n" "ds_read_b128 %13, %19 offset:2048\n"
            "ds_read_b128 %14, %19 offset:4096\n" "ds_read_b128 %15, %19 offset:6144\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(fw[0][0]), "=&v"(fw[0][1]), "=&v"(fw[0][2]), "=&v"(fw[0][3]),
              "=&v"(fa[0][0]), "=&v"(fa[0][1]), "=&v"(fa[0][2]), "=&v"(fa[0][3]),
              "=&v"(fw[1][0]), "=&v"(fw[1][1]), "=&v"(fw[1][2]), "=&v"(fw[1][3]),
              "=&v"(fa[1][0]), "=&v"(fa[1][1]), "=&v"(fa[1][2]), "=&v"(fa[1][3])
            : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
            : "memory");
      }
      if constexpr (TM == 2 && TN == 4) {
        asm volatile(
            "ds_read_b128 %0, %12 offset:0\n" "ds_read_b128 %1, %12 offset:2048\n"
            "ds_read_b128 %2, %12 offset:4096\n" "ds_read_b128 %3, %12 offset:6144\n"
            "ds_read_b128 %4, %14 offset:0\n" "ds_read_b128 %5, %14 offset:2048\n"
            "ds_read_b128 %6, %13 offset:0\n" "ds_read_b128 %7, %13 offset:2048\n"
            "ds_read_b128 %8, %13 offset:4096\n" "ds_read_b128 %9, %13 offset:6144\n"
            "ds_read_b128 %10, %15 offset:0\n" "ds_read_b128 %11, %15 offset:2048\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(fw[0][0]), "=&v"(fw[0][1]), "=&v"(fw[0][2]), "=&v"(fw[0][3]),
              "=&v"(fa[0][0]), "=&v"(fa[0][1]), "=&v"(fw[1][0]), "=&v"(fw[1][1]),
              "=&v"(fw[1][2]), "=&v"(fw[1][3]), "=&v"(fa[1][0]), "=&v"(fa[1][1])
            : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
            : "memory");
      }
      if constexpr (TM == 2 && TN == 2) {
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
      }
      if constexpr (TM == 1 && TN == 2) {
        asm volatile(
            "ds_read_b128 %0, %6 offset:0\n" "ds_read_b128 %1, %6 offset:2048\n"
            "ds_read_b128 %2, %8 offset:0\n" "ds_read_b128 %3, %7 offset:0\n"
            "ds_read_b128 %4, %7 offset:2048\n" "ds_read_b128 %5, %9 offset:0\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(fw[0][0]), "=&v"(fw[0][1]), "=&v"(fa[0][0]), "=&v"(fw[1][0]),
              "=&v"(fw[1][1]), "=&v"(fa[1][0])
            : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
            : "memory");
      }
    };
    auto multiply = [&]() {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[s][j], fa[s][i], acc[i][j], 0, 0, 0);
    };
    const int full = K / GG_BK;
#pragma unroll
    for (int i = 0; i < NS - 1; ++i)
      if (i < full) request(i * GG_BK, i);
    int p = 0, q = NS - 1;
    for (int step = 0; step < full; ++step) {
      // this step's tiles have arrived when only those requested after them are on their way
      if (step + NS - 2 < full) __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 2) * (LA + LW)));
      else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
      __builtin_amdgcn_s_barrier();
      take(p);
      if (step + NS - 1 < full) request((step + NS - 1) * GG_BK, q);
      multiply();
      __builtin_amdgcn_sched_barrier(0);     // (or the products move behind the next wait)
      p = p + 1 == NS ? 0 : p + 1;
      q = q + 1 == NS ? 0 : q + 1;
    }
    if (full * GG_BK < K) {      // the rest of a K that is no multiple of 64 (of 8, always)
      const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
      // (place p: the last reader of it was NS steps back, and no request for it is under way)
      const bool in = full * GG_BK + piece * 8 < K;
#pragma unroll
      for (int i = 0; i < LA; ++i)
        *reinterpret_cast<bf16x8_t*>(&As[p][(32 * i + wave * 8) * GG_BK + lane * 8]) =
            in ? *reinterpret_cast<const bf16x8_t*>(arow[i] + full * GG_BK) : zero8;
#pragma unroll
      for (int i = 0; i < LW; ++i)
        *reinterpret_cast<bf16x8_t*>(&Ws[p][(32 * i + wave * 8) * GG_BK + lane * 8]) =
            in ? *reinterpret_cast<const bf16x8_t*>(wrow[i] + full * GG_BK) : zero8;
      __syncthreads();
      take(p);
      multiply();
    }
  }
};
