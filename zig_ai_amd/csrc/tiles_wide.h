// Products of rows with rows, bfloat16 into 32-bit sums on the matrix cores, in tiles of 256, 192 or
// 128 rows of A x 256 rows of W: what a step of many rows is bound by, the matrix cores and the power
// that they and the ways to them take.
//
// Four waves, one a SIMD, two along the rows of A and two along those of W: a wave's part is 128 x 128
// (96 x 128, 64 x 128), its sums fill the accumulation registers, and an element read from LDS is
// multiplied 64 times.  With random operands the card's power bounds them: eight waves with 128 x 64 each, which
// read half as much again from LDS, take as many clocks a step, but ran at 1,550 MHz where these run at 1,620 to
// 1,700 (2,048 x 16,384 x 2,048; with zeros both run at 2,350).
//
// A phase is 32 elements of K.  It is made of blocks of 16 products, each one asm statement: the reads of
// the next phase's fragments and the requests from memory stand between the products, in their shadow,
// and the wait for the reads ends the statement, as their results may only be known to the compiler when
// they are there.  Two phases, 64 elements of K, are a step:
//
//   phase 0   multiplies the step's first half   reads its second half   requests W of step s + 2
//   wait for the tiles of step s + 1, barrier: the place of A(s) is free
//   phase 1   multiplies the second half         reads step s + 1's first half   requests A of step s + 2
//
// 2,250 clocks a step of 256 x 256, 2,048 of them products.  (W of step s + 3 requested with A, half a step
// earlier but four requests a block: 2,340.)  The tiles go from memory into LDS without passing registers, whole
// lines of 128 bytes, as in tiles_bf16.h (requests of 64 bytes a row halve what the second-level cache
// delivers); a request is a 32-bit offset a lane from a base in scalar registers.
// All that LDS holds is taken: three places for W, which comes from memory, and two for A, which an
// expert's or a layer's stretches of outputs share.  Operand layout and sums are those of tiles_bf16.h:
// K in steps of 32, in order.
#pragma once

#include "tiles_bf16.h"

#define GW_LDS (160 * 1024)      // bytes of a workgroup's LDS, all there is
#define GW_PLACE (256 * GG_BK * 2)

// ---- a block: 16 products of two rows of fragments of A with eight of W
#define GW_MF0(j) "v_mfma_f32_16x16x32_bf16 %[c" #j "], %[w" #j "], %[a0], %[c" #j "]\n"
#define GW_MF1(j) "v_mfma_f32_16x16x32_bf16 %[d" #j "], %[w" #j "], %[a1], %[d" #j "]\n"
#define GW_RD(k) "ds_read_b128 %[n" #k "], %[p" #k "] offset:%[o" #k "]\n"
// (one instruction ahead of the request, which needs that distance)
#define GW_TO(k) "s_mov_b32 m0, %[m" #k "]\n"
#define GW_RQ(k) "global_load_lds_dwordx4 %[v" #k "], %[from]\n"
// what stands behind the first to the fifteenth product
#define GW_TEXT(b0, b1, b2, b3, b4, b5, b6, b7, b8, b9, b10, b11, b12)                                                \
  GW_MF0(0) b0 GW_MF0(1) b1 GW_MF0(2) b2 GW_MF0(3) b3 GW_MF0(4) b4 GW_MF0(5) b5 GW_MF0(6) b6 GW_MF0(7) b7 GW_MF1(0) b8 \
  GW_MF1(1) b9 GW_MF1(2) b10 GW_MF1(3) b11 GW_MF1(4) b12 GW_MF1(5) GW_MF1(6) GW_MF1(7) "s_waitcnt lgkmcnt(0)\n"
#define GW_READS4 GW_RD(0), GW_RD(1), GW_RD(2), GW_RD(3)
#define GW_READS5 GW_READS4 GW_RD(4)
#define GW_READS6 GW_RD(0) GW_RD(4), GW_RD(1) GW_RD(5), GW_RD(2), GW_RD(3)
#define GW_NONE "", "", "", "", "", "", "", "", ""
#define GW_REQUESTS2 GW_TO(0), GW_RQ(0), "", "", GW_TO(1), GW_RQ(1), "", "", ""
#define GW_REQUESTS3 GW_TO(0), GW_RQ(0), "", GW_TO(1), GW_RQ(1), "", GW_TO(2), GW_RQ(2), ""
#define GW_REQUESTS4 GW_TO(0), GW_RQ(0), GW_TO(1), GW_RQ(1), GW_TO(2), GW_RQ(2), GW_TO(3), GW_RQ(3), ""
#define GW_CALL(f, ...) f(__VA_ARGS__)
#define GW_SUMS                                                                                              \
  [c0] "+a"(c[0]), [c1] "+a"(c[1]), [c2] "+a"(c[2]), [c3] "+a"(c[3]), [c4] "+a"(c[4]), [c5] "+a"(c[5]),           \
  [c6] "+a"(c[6]), [c7] "+a"(c[7]), [d0] "+a"(d[0]), [d1] "+a"(d[1]), [d2] "+a"(d[2]), [d3] "+a"(d[3]),           \
  [d4] "+a"(d[4]), [d5] "+a"(d[5]), [d6] "+a"(d[6]), [d7] "+a"(d[7])
#define GW_OUT(k) [n##k] "=&v"(*read[k].to)
#define GW_OUT4 GW_OUT(0), GW_OUT(1), GW_OUT(2), GW_OUT(3)
#define GW_OUT5 GW_OUT4, GW_OUT(4)
#define GW_OUT6 GW_OUT5, GW_OUT(5)
#define GW_PLACED(k) [p##k] "v"(read[k].at), [o##k] "n"(offset_of(FIRST + k))
#define GW_PLACED4 GW_PLACED(0), GW_PLACED(1), GW_PLACED(2), GW_PLACED(3)
#define GW_PLACED5 GW_PLACED4, GW_PLACED(4)
#define GW_PLACED6 GW_PLACED5, GW_PLACED(5)
#define GW_OPERANDS                                                                                          \
  [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]), [w4] "v"(w[4]), [w5] "v"(w[5]), [w6] "v"(w[6]), \
  [w7] "v"(w[7]), [a0] "v"(a0), [a1] "v"(a1)
#define GW_REQUEST(k) [v##k] "v"(offset[k]), [m##k] "s"(to + (k) * 4096)
#define GW_REQUEST2 , GW_REQUEST(0), GW_REQUEST(1), [from] "s"(from)
#define GW_REQUEST3 , GW_REQUEST(0), GW_REQUEST(1), GW_REQUEST(2), [from] "s"(from)
#define GW_REQUEST4 , GW_REQUEST(0), GW_REQUEST(1), GW_REQUEST(2), GW_REQUEST(3), [from] "s"(from)
#define GW_BLOCK(R, READS, REQUESTS, INPUTS)                                                          \
  asm volatile(GW_CALL(GW_TEXT, READS, REQUESTS) : GW_SUMS, GW_OUT##R : GW_OPERANDS, GW_PLACED##R INPUTS \
               : "memory", "m0")

template <int TM>      // a wave's rows of A in sixteens; the tile has 32 TM
struct TilesWide {
  static_assert(TM == 8 || TM == 6 || TM == 4, "see step");
  static constexpr int TN = 8, LA = TM, LW = 8;
  struct Read {
    bf16x8_t* to;
    unsigned at;
  };
  // fragment f of a phase, eight of W and then TM of A: its distance from the first of its operand
  static constexpr int offset_of(int f) { return (f < 8 ? f : f - 8) * 16 * GG_BK * 2; }

  // 16 products beside the reads of fragments FIRST .. FIRST + R - 1 and Q requests
  template <int FIRST, int R, int Q>
  static __device__ __forceinline__ void block(f32x4_t (&c)[TN], f32x4_t (&d)[TN], const bf16x8_t (&w)[8],
                                               const bf16x8_t& a0, const bf16x8_t& a1, const Read (&read)[R],
                                               const unsigned* offset, unsigned to, const char* from) {
    static_assert((R == 4 && (Q == 0 || Q == 2)) || (R == 5 && (Q == 0 || Q == 2 || Q == 3)) ||
                  (R == 6 && (Q == 0 || Q == 2 || Q == 4)), "see below");
    if constexpr (R == 4 && Q == 0) GW_BLOCK(4, GW_READS4, GW_NONE, );
    if constexpr (R == 4 && Q == 2) GW_BLOCK(4, GW_READS4, GW_REQUESTS2, GW_REQUEST2);
    if constexpr (R == 5 && Q == 0) GW_BLOCK(5, GW_READS5, GW_NONE, );
    if constexpr (R == 5 && Q == 2) GW_BLOCK(5, GW_READS5, GW_REQUESTS2, GW_REQUEST2);
    if constexpr (R == 5 && Q == 3) GW_BLOCK(5, GW_READS5, GW_REQUESTS3, GW_REQUEST3);
    if constexpr (R == 6 && Q == 0) GW_BLOCK(6, GW_READS6, GW_NONE, );
    if constexpr (R == 6 && Q == 2) GW_BLOCK(6, GW_READS6, GW_REQUESTS2, GW_REQUEST2);
    if constexpr (R == 6 && Q == 4) GW_BLOCK(6, GW_READS6, GW_REQUESTS4, GW_REQUEST4);
  }

  // A phase: products of `w` and `a`; `nw`, `na` take the fragments at `atw`, `ata`.  QW: W's tile is requested,
  // QA: A's.
  template <bool QW, bool QA>
  static __device__ __forceinline__ void phase(f32x4_t (&acc)[TM][TN], const bf16x8_t (&w)[8], const bf16x8_t (&a)[TM],
                                               bf16x8_t (&nw)[8], bf16x8_t (&na)[TM], unsigned atw, unsigned ata,
                                               const unsigned* offset, unsigned to, const char* from) {
#define GW_R(f) Read{(f) < 8 ? &nw[(f) & 7] : &na[(f) < 8 ? 0 : (f) - 8], (f) < 8 ? atw : ata}
    if constexpr (TM == 8) {
      constexpr int Q = QW || QA ? 2 : 0;
      block<0, 4, Q>(acc[0], acc[1], w, a[0], a[1], {GW_R(0), GW_R(1), GW_R(2), GW_R(3)}, offset, to, from);
      block<4, 4, Q>(acc[2], acc[3], w, a[2], a[3], {GW_R(4), GW_R(5), GW_R(6), GW_R(7)}, offset + 2, to + 8192, from);
      block<8, 4, Q>(acc[4], acc[5], w, a[4], a[5], {GW_R(8), GW_R(9), GW_R(10), GW_R(11)}, offset + 4, to + 16384, from);
      block<12, 4, Q>(acc[6], acc[7], w, a[6], a[7], {GW_R(12), GW_R(13), GW_R(14), GW_R(15)}, offset + 6, to + 24576, from);
    } else if constexpr (TM == 6) {
      constexpr int Q = QW ? 3 : QA ? 2 : 0, L = QW || QA ? 2 : 0;
      block<0, 5, Q>(acc[0], acc[1], w, a[0], a[1], {GW_R(0), GW_R(1), GW_R(2), GW_R(3), GW_R(4)}, offset, to, from);
      block<5, 5, Q>(acc[2], acc[3], w, a[2], a[3], {GW_R(5), GW_R(6), GW_R(7), GW_R(8), GW_R(9)}, offset + Q, to + Q * 4096, from);
      block<10, 4, L>(acc[4], acc[5], w, a[4], a[5], {GW_R(10), GW_R(11), GW_R(12), GW_R(13)}, offset + 2 * Q, to + 2 * Q * 4096, from);
    } else {
      constexpr int Q = QW ? 4 : QA ? 2 : 0;
      block<0, 6, Q>(acc[0], acc[1], w, a[0], a[1], {GW_R(0), GW_R(1), GW_R(2), GW_R(3), GW_R(4), GW_R(5)}, offset, to, from);
      block<6, 6, Q>(acc[2], acc[3], w, a[2], a[3], {GW_R(6), GW_R(7), GW_R(8), GW_R(9), GW_R(10), GW_R(11)}, offset + Q, to + Q * 4096, from);
    }
#undef GW_R
  }

  // `offa`, `offw`: bytes from `abase`, `wbase` to a lane's rows 32 i + 8 wave + lane / 8 of the tile, each
  // at its piece (lane % 8) ^ (lane / 8) of 16 bytes; K is a multiple of 64.  acc[i][j][r]: row
  // wm + 16 i + lane % 16 of A and wn + 16 j + lane / 16 * 4 + r of W, wm = (wave / 2) * 16 TM,
  // wn = (wave % 2) * 128.  `meanwhile` runs while the first tiles are on their way.  Other waves may still
  // read LDS when it returns.
  template <typename Meanwhile>
  static __device__ __forceinline__ void run(char (&lds)[GW_LDS], int wave, int lane, int K, const char* abase,
                                             const char* wbase, const unsigned (&offa)[LA], const unsigned (&offw)[LW],
                                             f32x4_t (&acc)[TM][TN], Meanwhile meanwhile) {
    const int steps = K / GG_BK;
    const unsigned As = lds_address(lds), Ws = As + 2 * GW_PLACE, own = wave * 1024;
    auto request = [&](const char* from, unsigned offset, unsigned to) {
      asm volatile("s_mov_b32 m0, %0\n" "s_nop 0\n" "global_load_lds_dwordx4 %1, %2\n"
                   :: "s"(to), "v"(offset), "s"(from) : "memory", "m0");
    };
    auto request_step = [&](int s) {
#pragma unroll
      for (int i = 0; i < LW; ++i) request(wbase + s * (GG_BK * 2), offw[i], Ws + s * GW_PLACE + own + i * 4096);
#pragma unroll
      for (int i = 0; i < LA; ++i) request(abase + s * (GG_BK * 2), offa[i], As + s * GW_PLACE + own + i * 4096);
    };
    auto meet = [&]() {      // nothing moves over it
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    request_step(0);
    if (steps > 1) request_step(1);
    meanwhile();
    // (clearing 256 registers takes 1,024 clocks: not behind the wait)
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]),
                   "+a"(acc[i][6]), "+a"(acc[i][7]));
    }
    if (steps > 1) __builtin_amdgcn_s_waitcnt(ZA_VMCNT(LA + LW));
    else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
    const int r16 = lane & 15, kq = lane >> 4;
    const unsigned half[2] = {(unsigned)((kq ^ (r16 & 7)) * 16), (unsigned)(((4 + kq) ^ (r16 & 7)) * 16)};
    const unsigned ra = As + ((wave >> 1) * 16 * TM + r16) * (GG_BK * 2);
    const unsigned rw = Ws + ((wave & 1) * 128 + r16) * (GG_BK * 2);
    bf16x8_t a0[TM], w0[8], a1[TM], w1[8];
    meet();
    {
      const unsigned w = rw + half[0], a = ra + half[0];
      asm volatile("ds_read_b128 %0, %8 offset:0\n" "ds_read_b128 %1, %8 offset:2048\n" "ds_read_b128 %2, %8 offset:4096\n"
                   "ds_read_b128 %3, %8 offset:6144\n" "ds_read_b128 %4, %8 offset:8192\n" "ds_read_b128 %5, %8 offset:10240\n"
                   "ds_read_b128 %6, %8 offset:12288\n" "ds_read_b128 %7, %8 offset:14336\n" "s_waitcnt lgkmcnt(0)"
                   : "=&v"(w0[0]), "=&v"(w0[1]), "=&v"(w0[2]), "=&v"(w0[3]), "=&v"(w0[4]), "=&v"(w0[5]), "=&v"(w0[6]), "=&v"(w0[7])
                   : "v"(w) : "memory");
#pragma unroll
      for (int i = 0; i < TM; i += 2)
        asm volatile("ds_read_b128 %0, %2 offset:0\n" "ds_read_b128 %1, %2 offset:2048\n" "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a0[i]), "=&v"(a0[i + 1]) : "v"(a + i * 2048) : "memory");
    }
    // places of W(s), W(s + 1), W(s + 2) and A(s), and what the requests for step s + 2 begin at
    unsigned pw = 0, pw1 = GW_PLACE, pw2 = 2 * GW_PLACE, pa = 0;
    const char *af = abase + 4 * GG_BK, *wf = wbase + 4 * GG_BK;
    auto step = [&](auto more) {
      constexpr bool MORE = decltype(more)::value;
      phase<MORE, false>(acc, w0, a0, w1, a1, rw + pw + half[1], ra + pa + half[1], offw, Ws + pw2 + own, wf);
      // (of what is under way only this phase's requests may be left)
      if (MORE) __builtin_amdgcn_s_waitcnt(ZA_VMCNT(LW));
      else __builtin_amdgcn_s_waitcnt(ZA_VMCNT(0));
      meet();
      phase<false, MORE>(acc, w1, a1, w0, a0, rw + pw1 + half[0], ra + (pa ^ GW_PLACE) + half[0], offa, As + pa + own, af);
      const unsigned free = pw;
      pw = pw1;
      pw1 = pw2;
      pw2 = free;
      pa ^= GW_PLACE;
      af += GG_BK * 2;
      wf += GG_BK * 2;
    };
    int s = 0;
    for (; s + 2 < steps; ++s) step(std::true_type{});
    for (; s < steps; ++s) step(std::false_type{});      // (the last one's second reads find older tiles: not used)
    // the last products' sums may be read by other instructions only so many clocks later
    asm volatile("s_nop 15\n" "s_nop 15"
                 : "+a"(acc[TM - 1][0]), "+a"(acc[TM - 1][1]), "+a"(acc[TM - 1][2]), "+a"(acc[TM - 1][3]), "+a"(acc[TM - 1][4]),
                   "+a"(acc[TM - 1][5]), "+a"(acc[TM - 1][6]), "+a"(acc[TM - 1][7]));
#pragma unroll
    for (int i = 0; i < TM - 1; ++i)
      asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]),
                   "+a"(acc[i][6]), "+a"(acc[i][7]));
  }
};

// A tile's way out: 32-bit sums straight from their registers, 16 bytes a lane (through LDS, 47 us instead of
// 44: 7,108 rows, 2,048 x 1,024).  bfloat16 passes through a wave's 32 KB of LDS, so that what it stores are
// whole stretches of COLS outputs, 16 bytes a lane (from the registers, 8 bytes of sixteen rows an
// instruction, a tile of 256 x 256 took 15,900 clocks instead of 7,200).
//   fill(i, j)   outputs 16 j + lane / 16 * 4 .. + 3 of the wave's row 16 i + lane % 16
//   row_at(i, r) the row of `out` that the wave's row 16 i + r goes to, or less than 0; all lanes ask, in 32 bits
//                each for its own row of the sums' layout
// `n` is the wave's first column of the N of a row.  All waves have passed a barrier behind their last
// read of LDS.
template <typename TO, int COLS, int TM, typename Fill, typename RowAt>
__device__ __forceinline__ void wide_store(char (&lds)[GW_LDS], int wave, int lane, TO* out, int n, int N, Fill fill,
                                           RowAt row_at) {
  const int r16 = lane & 15, kq = lane >> 4;
  constexpr int EACH = 16 / (int)sizeof(TO);      // elements a store
  const bool whole = N % EACH == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0, inside = whole && n + COLS <= N;
  auto put = [&](TO* row, int at, auto from) {     // EACH elements from column `at` on
    if (inside) {
      *reinterpret_cast<decltype(from)*>(row + at) = from;
    } else if (whole) {
      if (at < N) *reinterpret_cast<decltype(from)*>(row + at) = from;
    } else {
#pragma unroll
      for (int e = 0; e < EACH; ++e)
        if (at + e < N) row[at + e] = from[e];
    }
  };
  if constexpr (sizeof(TO) == 4) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int to = row_at(i, r16);
      if (to < 0) continue;
      TO* row = out + (size_t)to * N;
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j) put(row, n + 16 * j + 4 * kq, fill(i, j));
    }
  } else {
    constexpr int PIECES = COLS / 8, AT_ONCE = 64 / PIECES;      // 16 bytes each, in a row; rows an instruction
    bf16_t* own = reinterpret_cast<bf16_t*>(lds + wave * 32768);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = 16 * i + r16;
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j) {
        const f32x4_t v = fill(i, j);
        *reinterpret_cast<bf16x4_t*>(own + row * COLS + ((2 * j + (kq >> 1)) ^ (row & (PIECES - 1))) * 8 + (kq & 1) * 4) =
            bf16x4_t{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < TM * 16 / AT_ONCE; ++t) {
      const int row = t * AT_ONCE + lane / PIECES, piece = lane % PIECES;
      const int to = row_at(t * AT_ONCE / 16, t * AT_ONCE % 16 + lane / PIECES);
      const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(own + row * COLS + (piece ^ (row & (PIECES - 1))) * 8);
      if (to >= 0) put(out + (size_t)to * N, n + piece * 8, v);
    }
  }
}
