// Products of rows with rows, bfloat16 into 32-bit sums on the matrix cores, in tiles of 256, 192 or 128 rows
// of A x 128 rows of W: where tiles of 256 x 256 (tiles_wide.h) would leave compute units idle.
//
// Four waves, one a SIMD, two along the rows of A and two along those of W: a wave's part is 128 x 64 (96 x 64,
// 64 x 64).  Phases, blocks and steps are those of tiles_wide.h: reads of the next phase's fragments and requests
// from memory in the products' shadow, one barrier a step.  A step's tiles lie in one of NS places (three to
// five, 144 to 160 KB of LDS); a place is requested for from the barrier on behind which it is free:
//
//   phase 0   multiplies the step's first half   reads its second half   requests W of step s + NS - 1
//   wait for the tiles of step s + 1, barrier: the place of step s is free
//   phase 1   multiplies the second half         reads step s + 1's first half   requests A of step s + NS
//
// LDS bounds it where the wide tiles are bound by the matrix cores: a step takes (96 TM + 384) clocks of LDS and
// 128 TM of products.
#pragma once

#include "tiles_wide.h"

#define GH_MF(i, j) "v_mfma_f32_16x16x32_bf16 %[c" #i #j "], %[w" #j "], %[a" #i "], %[c" #i #j "]\n"
#define GH_ROW(i, b0, b1, b2, b3) GH_MF(i, 0) b0 GH_MF(i, 1) b1 GH_MF(i, 2) b2 GH_MF(i, 3) b3
#define GH_WAIT "s_waitcnt lgkmcnt(0)\n"
#define GH_SUMS_OF(i) \
  [c##i##0] "+a"(c[i][0]), [c##i##1] "+a"(c[i][1]), [c##i##2] "+a"(c[i][2]), [c##i##3] "+a"(c[i][3])
#define GH_SUMS3 GH_SUMS_OF(0), GH_SUMS_OF(1), GH_SUMS_OF(2)
#define GH_SUMS4 GH_SUMS3, GH_SUMS_OF(3)
#define GH_OUT8 GW_OUT6, GW_OUT(6), GW_OUT(7)
#define GH_PLACED8 GW_PLACED6, GW_PLACED(6), GW_PLACED(7)
#define GH_W [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3])
#define GH_IN3 GH_W, [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2])
#define GH_IN4 GH_IN3, [a3] "v"(a[3])
#define GH_BLOCK(TEXT, R, READS, ...) \
  asm volatile(TEXT GH_WAIT : GH_SUMS##R, READS : GH_IN##R, __VA_ARGS__ : "memory", "m0")
#define GH_RQ2 GW_REQUEST(0), GW_REQUEST(1), [from] "s"(from)
#define GH_RQ3 GW_REQUEST(0), GW_REQUEST(1), GW_REQUEST(2), [from] "s"(from)
#define GH_RQ4 GW_REQUEST(0), GW_REQUEST(1), GW_REQUEST(2), GW_REQUEST(3), [from] "s"(from)

template <int TM>      // a wave's rows of A in sixteens; the tile has 32 TM
struct TilesHalf {
  static_assert(TM == 8 || TM == 6 || TM == 4, "see phase");
  static constexpr int TN = 4, LA = TM, LW = 4, NS = TM == 8 ? 3 : TM == 6 ? 4 : 5;
  static constexpr int ROWS = TM == 6 ? 3 : 4, BLOCKS = TM / ROWS;      // of fragments a block, blocks a phase
  static constexpr int PLACE = (32 * TM + 128) * GG_BK * 2;             // W's rows behind A's
  static_assert(NS * PLACE <= GW_LDS, "LDS");
  struct Read {
    bf16x8_t* to;
    unsigned at;
  };
  // fragment f of a phase, four of W and then TM of A: its distance from the first of its operand
  static constexpr int offset_of(int f) { return (f < 4 ? f : f - 4) * 16 * GG_BK * 2; }

  // 4 ROWS products beside the reads of fragments FIRST .. FIRST + R - 1 and Q requests
  template <int FIRST, int R, int Q>
  static __device__ __forceinline__ void block(f32x4_t (*c)[TN], const bf16x8_t (&w)[4], const bf16x8_t* a,
                                               const Read (&read)[R], const unsigned* offset, unsigned to,
                                               const char* from) {
    if constexpr (ROWS == 4 && R == 6 && Q == 0)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4), GW_RD(5), , ) GH_ROW(2, , , , )
               GH_ROW(3, , , , ), 4, GW_OUT6, GW_PLACED6);
    if constexpr (ROWS == 4 && R == 6 && Q == 2)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4), GW_RD(5) GW_TO(0), GW_RQ(0), )
               GH_ROW(2, , GW_TO(1), GW_RQ(1), ) GH_ROW(3, , , , ), 4, GW_OUT6, GW_PLACED6, GH_RQ2);
    if constexpr (ROWS == 4 && R == 6 && Q == 4)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4), GW_RD(5) GW_TO(0), GW_RQ(0), GW_TO(1))
               GH_ROW(2, GW_RQ(1), GW_TO(2), GW_RQ(2), GW_TO(3)) GH_ROW(3, GW_RQ(3), , , ), 4, GW_OUT6, GW_PLACED6, GH_RQ4);
    if constexpr (ROWS == 4 && R == 8 && Q == 0)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4), GW_RD(5), GW_RD(6), GW_RD(7))
               GH_ROW(2, , , , ) GH_ROW(3, , , , ), 4, GH_OUT8, GH_PLACED8);
    if constexpr (ROWS == 4 && R == 8 && Q == 4)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2) GW_TO(0), GW_RD(3) GW_RQ(0))
               GH_ROW(1, GW_RD(4) GW_TO(1), GW_RD(5) GW_RQ(1), GW_RD(6), GW_RD(7)) GH_ROW(2, GW_TO(2), GW_RQ(2), , GW_TO(3))
               GH_ROW(3, GW_RQ(3), , , ), 4, GH_OUT8, GH_PLACED8, GH_RQ4);
    if constexpr (ROWS == 3 && R == 5 && Q == 0)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4), , , ) GH_ROW(2, , , , ), 3, GW_OUT5,
               GW_PLACED5);
    if constexpr (ROWS == 3 && R == 5 && Q == 2)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4) GW_TO(0), GW_RQ(0), , GW_TO(1))
               GH_ROW(2, GW_RQ(1), , , ), 3, GW_OUT5, GW_PLACED5, GH_RQ2);
    if constexpr (ROWS == 3 && R == 5 && Q == 3)
      GH_BLOCK(GH_ROW(0, GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)) GH_ROW(1, GW_RD(4) GW_TO(0), GW_RQ(0), GW_TO(1), GW_RQ(1))
               GH_ROW(2, GW_TO(2), GW_RQ(2), , ), 3, GW_OUT5, GW_PLACED5, GH_RQ3);
  }

  struct Requests {      // offsets of A's TM rows and W's four behind them, where to, and A's and W's base
    const unsigned* offset;
    unsigned to;
    const char *a, *w;
  };
  // A phase: products of `w` and `a`; `nw`, `na` take the fragments at `atw`, `ata`.  MORE: it requests, in the
  // SECOND phase A's tile, else W's.
  template <bool SECOND, bool MORE>
  static __device__ __forceinline__ void phase(f32x4_t (&acc)[TM][TN], const bf16x8_t (&w)[4], const bf16x8_t (&a)[TM],
                                               bf16x8_t (&nw)[4], bf16x8_t (&na)[TM], unsigned atw, unsigned ata,
                                               const Requests& q) {
#define GH_R(f) Read{(f) < 4 ? &nw[(f) & 3] : &na[(f) < 4 ? 0 : (f) - 4], (f) < 4 ? atw : ata}
#define GH_Q(i) q.offset + (i), q.to + (i) * 4096, (i) < LA ? q.a : q.w
    if constexpr (TM == 8) {      // 12 requests: A's eight, W's four
      constexpr int Q0 = !MORE ? 0 : SECOND ? 4 : 2;
      block<0, 6, Q0>(acc, w, a, {GH_R(0), GH_R(1), GH_R(2), GH_R(3), GH_R(4), GH_R(5)}, GH_Q(SECOND ? 0 : 8));
      block<6, 6, Q0>(acc + 4, w, a + 4, {GH_R(6), GH_R(7), GH_R(8), GH_R(9), GH_R(10), GH_R(11)}, GH_Q(SECOND ? 4 : 10));
    } else if constexpr (TM == 6) {      // 10: A's six, W's four
      constexpr int Q = !MORE ? 0 : SECOND ? 3 : 2;
      block<0, 5, Q>(acc, w, a, {GH_R(0), GH_R(1), GH_R(2), GH_R(3), GH_R(4)}, GH_Q(SECOND ? 0 : 6));
      block<5, 5, Q>(acc + 3, w, a + 3, {GH_R(5), GH_R(6), GH_R(7), GH_R(8), GH_R(9)}, GH_Q(SECOND ? 3 : 8));
    } else {      // 8: A's four, W's four
      block<0, 8, MORE ? 4 : 0>(acc, w, a, {GH_R(0), GH_R(1), GH_R(2), GH_R(3), GH_R(4), GH_R(5), GH_R(6), GH_R(7)},
                                GH_Q(SECOND ? 0 : 4));
    }
#undef GH_R
#undef GH_Q
  }

  // As TilesWide's, but `off` are A's TM offsets and W's four behind them, wn = (wave % 2) * 64, and K is at least
  // NS steps.
  static __device__ __forceinline__ void run(char (&lds)[GW_LDS], int wave, int lane, int K, const char* abase,
                                             const char* wbase, const unsigned (&off)[LA + LW], f32x4_t (&acc)[TM][TN]) {
    const int steps = K / GG_BK;
    const unsigned base = lds_address(lds), own = wave * 1024;
    auto request = [&](const char* from, unsigned offset, unsigned to) {
      asm volatile("s_mov_b32 m0, %0\n" "s_nop 0\n" "global_load_lds_dwordx4 %1, %2\n"
                   :: "s"(to), "v"(offset), "s"(from) : "memory", "m0");
    };
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int i = 0; i < (s < NS - 1 ? LA + LW : LA); ++i)
        request((i < LA ? abase : wbase) + s * (GG_BK * 2), off[i], base + s * PLACE + own + i * 4096);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]));
    }
    auto meet = [&]() {      // nothing moves over it
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    const int r16 = lane & 15, kq = lane >> 4;
    const unsigned half[2] = {(unsigned)((kq ^ (r16 & 7)) * 16), (unsigned)(((4 + kq) ^ (r16 & 7)) * 16)};
    const unsigned ra = base + ((wave >> 1) * 16 * TM + r16) * (GG_BK * 2);
    const unsigned rw = base + (32 * TM + (wave & 1) * 64 + r16) * (GG_BK * 2);
    __builtin_amdgcn_s_waitcnt(ZA_VMCNT((NS - 2) * (LA + LW) + LA));
    meet();
    bf16x8_t a0[TM], w0[4], a1[TM], w1[4];
    {
      const unsigned w = rw + half[0], a = ra + half[0];
      asm volatile("ds_read_b128 %0, %4 offset:0\n" "ds_read_b128 %1, %4 offset:2048\n" "ds_read_b128 %2, %4 offset:4096\n"
                   "ds_read_b128 %3, %4 offset:6144\n" "s_waitcnt lgkmcnt(0)"
                   : "=&v"(w0[0]), "=&v"(w0[1]), "=&v"(w0[2]), "=&v"(w0[3]) : "v"(w) : "memory");
#pragma unroll
      for (int i = 0; i < TM; i += 2)
        asm volatile("ds_read_b128 %0, %2 offset:0\n" "ds_read_b128 %1, %2 offset:2048\n" "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a0[i]), "=&v"(a0[i + 1]) : "v"(a + i * 2048) : "memory");
    }
    // the places of step s and of the ones after and before it, and what its latest requests begin at
    unsigned at = 0, next = PLACE, before = (NS - 1) * PLACE;
    Requests q{off, 0, abase + NS * (GG_BK * 2), wbase + (NS - 1) * (GG_BK * 2)};
    // LATE: how many whole steps behind s + 1 are under way at the barrier, with W of the last
    auto step = [&](auto w_too, auto a_too, auto late) {
      q.to = base + before + own;
      phase<false, decltype(w_too)::value>(acc, w0, a0, w1, a1, rw + at + half[1], ra + at + half[1], q);
      __builtin_amdgcn_s_waitcnt(ZA_VMCNT(decltype(late)::value * (LA + LW)));
      meet();
      q.to = base + at + own;
      // (the last step's reads find an older step's tiles: not used)
      phase<true, decltype(a_too)::value>(acc, w1, a1, w0, a0, rw + next + half[0], ra + next + half[0], q);
      before = at;
      at = next;
      next = next == (NS - 1) * PLACE ? 0 : next + PLACE;
      q.a += GG_BK * 2;
      q.w += GG_BK * 2;
    };
    constexpr auto yes = std::true_type{};
    constexpr auto no = std::false_type{};
    for (int s = 0; s + NS < steps; ++s) step(yes, yes, std::integral_constant<int, NS - 2>{});
    step(yes, no, std::integral_constant<int, NS - 2>{});
    step(no, no, std::integral_constant<int, NS - 3>{});
    if constexpr (NS > 3) step(no, no, std::integral_constant<int, (NS > 3 ? NS - 4 : 0)>{});
    if constexpr (NS > 4) step(no, no, std::integral_constant<int, (NS > 4 ? NS - 5 : 0)>{});
    step(no, no, std::integral_constant<int, 0>{});
    // the last products' sums may be read by other instructions only so many clocks later
    asm volatile("s_nop 15\n" "s_nop 15" : "+a"(acc[TM - 1][0]), "+a"(acc[TM - 1][1]), "+a"(acc[TM - 1][2]), "+a"(acc[TM - 1][3]));
#pragma unroll
    for (int i = 0; i < TM - 1; ++i) asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]));
  }
};
