// Products of rows with rows, bfloat16 into 32-bit sums on the matrix cores, in tiles of 256 or 128
// rows of A x 256 rows of W: what a step of many rows is bound by, the matrix cores themselves.
//
// Eight waves, two a SIMD: waves 0 to 3 take the upper half of A's rows, 4 to 7 the lower, each 64
// rows of W (a wave's part is 128 x 64 or 64 x 64, so that an element read from LDS is multiplied
// 43 or 32 times; with 64 x 64 of 128 x 128 the reads and the tiles' way into LDS took half as long
// again as the products).  The halves are one slot apart: while one multiplies its 32 elements of K
// (a phase), the other, on the same SIMDs, reads its fragments of a phase, and a barrier ends the slot.
//
//   slot 2p      upper: multiplies phase p          lower: reads phase p
//   slot 2p + 1  upper: reads phase p + 1           lower: multiplies phase p
//
// The tiles go from memory into LDS without passing registers, 64 elements of K (two phases) a step, as
// in tiles_bf16.h: whole lines of 128 bytes (requests of 64 bytes a row, 32 elements, halve what the
// second-level cache delivers).  A half requests only in slots in which it reads: a request keeps a wave
// some 65 clocks, in front of its products or in their midst that is time the matrix cores stand still
// (2,970 clocks a step; 2,290 as it is, 2,048 of them products).  All that LDS holds is taken: three
// places for W, which comes from memory, and two for 256 rows of A, which an expert's stretches of
// outputs share, three for 128.
// Operand layout and sums are those of tiles_bf16.h: K in steps of 32, in order.
#pragma once

#include "tiles_bf16.h"

#define GW_LDS (160 * 512)      // elements of a workgroup's LDS, all there is

template <int TM>      // A's rows: 32 TM
struct TilesWide {
  static_assert(TM == 8 || TM == 4, "see take");
  static constexpr int TN = 4, LA = TM / 2, LW = 4;
  static constexpr int AP = TM == 8 ? 2 : 3, WP = 3;      // places of A and of W
  static constexpr int APLACE = 32 * TM * GG_BK, WPLACE = 256 * GG_BK;
  static_assert(AP * APLACE + WP * WPLACE <= GW_LDS, "LDS");

  // `arow`, `wrow`: a lane's rows 64 i + 8 wave + lane / 8 of the tile, each at its piece
  // (lane % 8) ^ (lane / 8) of 8 elements; K is a multiple of 64.  acc[i][j][r]: row
  // wm + 16 i + lane % 16 of A and wn + 16 j + lane / 16 * 4 + r of W, wm = (wave / 4) * 16 TM,
  // wn = (wave % 4) * 64.
  static __device__ __forceinline__ void run(bf16_t (&lds)[GW_LDS], int wave, int lane, int K,
                                             const bf16_t* const (&arow)[LA], const bf16_t* const (&wrow)[LW],
                                             f32x4_t (&acc)[TM][TN]) {
    const int steps = K / GG_BK;
    bf16_t *As = lds, *Ws = lds + AP * APLACE;
    // (nothing is requested beyond the last step)
    auto request_a = [&](int s, int place) {
      if (s >= steps) return;
#pragma unroll
      for (int i = 0; i < LA; ++i) lds_request(arow[i] + s * GG_BK, As + place * APLACE + (64 * i + 8 * wave) * GG_BK);
    };
    auto request_w = [&](int s, int place) {
      if (s >= steps) return;
#pragma unroll
      for (int i = 0; i < LW; ++i) lds_request(wrow[i] + s * GG_BK, Ws + place * WPLACE + (64 * i + 8 * wave) * GG_BK);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int r16 = lane & 15, kq = lane >> 4;
    const unsigned slot[2] = {(unsigned)((kq ^ (r16 & 7)) * 16), (unsigned)(((4 + kq) ^ (r16 & 7)) * 16)};
    const unsigned abase = lds_address(As + ((wave >> 2) * 16 * TM + r16) * GG_BK);
    const unsigned wbase = lds_address(Ws + ((wave & 3) * 64 + r16) * GG_BK);
    bf16x8_t fa[TM], fw[TN];
    // the fragments of one phase (the wait inside the block: see tiles_bf16.h)
    auto take = [&](int pa, int pw, int h) {
      const unsigned a = abase + pa * (APLACE * 2) + slot[h], w = wbase + pw * (WPLACE * 2) + slot[h];
      if constexpr (TM == 8) {
        asm volatile(
            "ds_read_b128 %0, %13 offset:0\n" "ds_read_b128 %1, %13 offset:2048\n"
            "ds_read_b128 %2, %13 offset:4096\n" "ds_read_b128 %3, %13 offset:6144\n"
            "ds_read_b128 %4, %12 offset:0\n" "ds_read_b128 %5, %12 offset:2048\n"
            "ds_read_b128 %6, %12 offset:4096\n" "ds_read_b128 %7, %12 offset:6144\n"
            "ds_read_b128 %8, %12 offset:8192\n" "ds_read_b128 %9, %12 offset:10240\n"
            "ds_read_b128 %10, %12 offset:12288\n" "ds_read_b128 %11, %12 offset:14336\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3]), "=&v"(fa[0]), "=&v"(fa[1]),
              "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fa[4]), "=&v"(fa[5]), "=&v"(fa[6]), "=&v"(fa[7])
            : "v"(a), "v"(w)
            : "memory");
      } else {
        asm volatile(
            "ds_read_b128 %0, %9 offset:0\n" "ds_read_b128 %1, %9 offset:2048\n"
            "ds_read_b128 %2, %9 offset:4096\n" "ds_read_b128 %3, %9 offset:6144\n"
            "ds_read_b128 %4, %8 offset:0\n" "ds_read_b128 %5, %8 offset:2048\n"
            "ds_read_b128 %6, %8 offset:4096\n" "ds_read_b128 %7, %8 offset:6144\n"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3]), "=&v"(fa[0]), "=&v"(fa[1]),
              "=&v"(fa[2]), "=&v"(fa[3])
            : "v"(a), "v"(w)
            : "memory");
      }
    };
    auto multiply = [&]() {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[j], fa[i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    // a slot's end; nothing moves over it
    auto meet = [&]() {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    // step s + 1 has arrived when only what was requested for s + 2 (of A with two places: W alone) is under way
    auto arrived = [&](int s) {
      if (s + 2 < steps) __builtin_amdgcn_s_waitcnt(ZA_VMCNT(AP == 3 ? LA + LW : LW));
      else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
    };
    // places: step % 2 or step % 3; `at` is s % 3, `next` (s + 1) % 3, `last` (s + 2) % 3
    auto after = [](int place) { return place == 2 ? 0 : place + 1; };
    request_w(0, 0);
    request_a(0, 0);
    request_w(1, 1);
    request_a(1, 1);
    if (AP == 3) request_w(2, 2);
    if (2 < steps) __builtin_amdgcn_s_waitcnt(ZA_VMCNT(LW + LA + (AP == 3 ? LW : 0)));
    else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
    meet();
    int at = 0;
    if (wave < 4) {
      take(0, 0, 0);
      for (int s = 0; s < steps; ++s) {
        const int next = after(at), last = after(next);
        const int pa = AP == 3 ? at : s & 1;
        meet();                                   // slot 4 s
        multiply();
        meet();
        if (AP == 3) request_a(s + 2, last);
        else request_w(s + 2, last);
        take(pa, at, 1);
        meet();
        multiply();
        __builtin_amdgcn_sched_barrier(0);
        arrived(s);
        meet();                                   // slot 4 s + 3
        if (AP == 3) request_w(s + 3, at);
        else request_a(s + 2, pa);
        if (s + 1 < steps) take(AP == 3 ? next : pa ^ 1, next, 0);
        at = next;
      }
    } else {
      for (int s = 0; s < steps; ++s) {
        const int next = after(at), last = after(next);
        const int pa = AP == 3 ? at : s & 1;
        meet();
        if (s > 0) {
          if (AP == 3) request_w(s + 2, last);
          else request_a(s + 1, pa ^ 1);
        }
        take(pa, at, 0);
        meet();
        multiply();
        meet();
        if (AP == 3) request_a(s + 2, last);
        else request_w(s + 2, last);
        take(pa, at, 1);
        arrived(s);
        meet();
        multiply();
        at = next;
      }
    }
  }
};
