// Attention over latent rows with every head's keys and values formed: for steps of long prompt
// portions.  latent.hip folds Wuk into the query and applies Wuv to the result, so a pair of query and
// key costs a head 2 x (2 R + Dr) operations (2,176 at R = 512 with 64 rotated); formed keys and
// values cost 2 x (d + Dr + dv) a pair (640 at heads of 128) and 2 R (d + dv) a key once, which
// is what folding and expanding cost a query.  So keys are formed where many new tokens see them.
//   latent_open_rows      the visible rows of every request, one request's behind the other's, out of
//                         the paged cache: the latents and the rotated key parts; the queries'
//                         rotated parts turned where they are
//   (a product of latents and [Wuk | Wuv]: all heads' keys, then all heads' values)
//   latent_expanded       the attention itself, with the gate in its epilogue
#include <math.h>

#include "attention_common.h"

#define LX_ROWS 64       // query rows of a work item, of one head
#define LX_KT 64         // keys of a tile
#define LX_D 128         // channels of a value and of a key without its rotated part

// ------------------------------------------------------------------ rows and rotation
struct OpenRowsArgs {
  bf16_t* q;                 // [T][H][q_ld]: elements q_col .. + Dr are turned in place
  int q_ld, q_col, H, Dr;
  const int* positions;      // [T]
  const float* inv_freq;
  int rot_dims, adjacent;
  float magnitude;
  unsigned pairs, pair_blocks;      // T * H * rot_dims / 2, and the workgroups that take them
  const bf16_t* plane;
  long long page_stride;
  const int* block_table;
  int bt_stride, page_size;
  const int* seq_start;      // [n_seqs + 1]
  const int* ctx_len;        // [n_seqs]
  int n_seqs, n_rows, R;
  bf16_t* latent;            // [n_rows][R]
  bf16_t* rot;               // [n_rows][Dr]
};

// A thread a pair of the queries; a wave a row of the cache (a row whose page is gone: zeros).
__global__ void __launch_bounds__(256)
latent_open_rows_kernel(OpenRowsArgs a) {
  if (blockIdx.x < a.pair_blocks) {
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= a.pairs) return;
    const unsigned half = a.rot_dims / 2, th = idx / half, i = idx % half;
    bf16_t* x = a.q + (size_t)th * a.q_ld + a.q_col;
    const unsigned u_at = a.adjacent ? 2 * i : i, v_at = a.adjacent ? 2 * i + 1 : i + half;
    float sn, cs;
    sincosf((float)a.positions[th / a.H] * a.inv_freq[i], &sn, &cs);
    sn *= a.magnitude;
    cs *= a.magnitude;
    const float u = (float)x[u_at], v = (float)x[v_at];
    x[u_at] = (bf16_t)(u * cs - v * sn);
    x[v_at] = (bf16_t)(v * cs + u * sn);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int row = (blockIdx.x - a.pair_blocks) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= a.n_rows) return;
  // whose row it is: requests' lengths added up, 64 at a time
  int before = 0;
  for (int s0 = 0; s0 < a.n_seqs; s0 += 64) {
    const int s = s0 + lane;
    const int len = s < a.n_seqs ? a.ctx_len[s] + a.seq_start[s + 1] - a.seq_start[s] : 0;
    int upto = len;
#pragma unroll
    for (int o = 1; o < ZA_WAVE; o <<= 1) {
      const int x = __shfl_up(upto, o, ZA_WAVE);
      if (lane >= o) upto += x;
    }
    const unsigned long long behind = __ballot(row < before + upto);
    if (behind == 0) {
      before += __shfl(upto, 63, ZA_WAVE);
      continue;
    }
    const int first = __builtin_ctzll(behind);
    const int place = row - before - (__shfl(upto, first, ZA_WAVE) - __shfl(len, first, ZA_WAVE));
    const int page = a.block_table[(size_t)(s0 + first) * a.bt_stride + place / a.page_size];
    const bf16_t* from = a.plane + (long long)max(page, 0) * a.page_stride + (long long)(place % a.page_size) * (a.R + a.Dr);
    for (int p = lane * 8; p < a.R + a.Dr; p += 512) {
      bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(from + p);
      if (page < 0) v = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
      bf16_t* to = p < a.R ? a.latent + (size_t)row * a.R + p : a.rot + (size_t)row * a.Dr + (p - a.R);
      *reinterpret_cast<bf16x8_t*>(to) = v;
    }
    return;
  }
}

// n_rows: the sum of ctx_len and the step's tokens, or more; rot_dims may be smaller than Dr.
extern "C" int za_latent_open_rows(void* q, int q_ld, int q_col, int n_tokens, int H, int Dr, const int* positions,
                                   const float* inv_freq, int rot_dims, int adjacent, float magnitude,
                                   const void* plane, long long page_stride, const int* block_table, int bt_stride,
                                   int page_size, const int* seq_start, const int* ctx_len, int n_seqs, int n_rows,
                                   int R, void* latent, void* rot, hipStream_t stream) {
  if (n_tokens == 0 || n_rows == 0) return 0;
  if (n_tokens < 0 || n_rows < 0 || H <= 0 || Dr < 0 || R <= 0 || n_seqs <= 0 || page_size <= 0 || bt_stride <= 0 ||
      rot_dims < 0 || rot_dims > Dr || rot_dims % 2 || q_col < 0 || q_col + Dr > q_ld || !q || !positions || !plane ||
      !block_table || !seq_start || !ctx_len || !latent || (Dr > 0 && !rot) || (rot_dims > 0 && !inv_freq) ||
      page_stride < (long long)page_size * (R + Dr))
    return ZA_ERR_ARG;
  if (R % 8 || Dr % 8 || page_stride % 8 ||
      ((reinterpret_cast<uintptr_t>(plane) | reinterpret_cast<uintptr_t>(latent) | reinterpret_cast<uintptr_t>(rot)) & 15))
    return ZA_ERR_UNSUPPORTED;
  const long long pairs = (long long)n_tokens * H * (rot_dims / 2);
  const long long pair_blocks = (pairs + 255) / 256, blocks = pair_blocks + ((long long)n_rows + 3) / 4;
  if (pairs + 256 > 0xffffffffLL || blocks > 0x7fffffffLL) return ZA_ERR_UNSUPPORTED;
  const OpenRowsArgs a{(bf16_t*)q, q_ld, q_col, H, Dr, positions, inv_freq, rot_dims, adjacent, magnitude,
                       (unsigned)pairs, (unsigned)pair_blocks, (const bf16_t*)plane, page_stride, block_table,
                       bt_stride, page_size, seq_start, ctx_len, n_seqs, n_rows, R, (bf16_t*)latent, (bf16_t*)rot};
  hipLaunchKernelGGL(latent_open_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return za_launch_status();
}

// ------------------------------------------------------------------------ attention
// A workgroup of four waves takes up to 64 tokens of one head, 16 rows a wave.  As in paged_attention_mfma_kernel:
//   S^T = K Q^T        queries in registers, keys from LDS; a lane has the scores of one row
//   p = 2^(S^T scale log2(e) - m), rounded to bfloat16; m the running maximum, not rounded: the largest
//                      weight is one, and rounding it to bfloat16 costs nothing
//   O^T += V^T P^T     P from the accumulator straight into the second operand; V^T from LDS, where values lie as
//                      they come, turned round on the way to registers (ds_read_b64_tr_b16)
// The next tile goes from memory into the other of two places in LDS without registers while one is computed.  A
// key's 16-byte pieces lie in the order piece ^ (key % 8), a value's piece ^ 2 (key % 8): the eight keys and the four
// values that are read together fall into different banks.
// What bounds it is the chain of a wave's tiles: the last rows of one prompt of 1,777 tokens see 28, and 448 workgroups
// leave a SIMD one or two waves.  So the fragments of a step are requested ahead of the products of the step before
// (left alone the compiler reads one, waits, and takes its product: 1.5 us a tile of 64 keys, 1.1 so), a step's products
// go to different accumulators, and a workgroup takes 64 rows and not 128 (1.4 us a tile for twice the rows: 47 us
// at 1,777 tokens where this takes 40; at 4,096 tokens 111 and 116).  Scores of the next tile beside the weights of this
// one, or a third place in LDS, gain nothing.
// 16 heads, R = 512 with 64 rotated, us with folding, expanding, rotating and gathering, folded (latent.hip) and
// formed: prompts of 512 tokens 61 and 36, 1,024 94 and 41, 1,777 149 and 62, 4,096 538 and 150; 512 tokens behind
// 1,000 cached ones 111 and 50, 256 behind 2,000 145 and 67.  Its error against 64 bits is that of the folded form within a
// twentieth, less behind cached rows (2.6e-3 for 3.1e-3 of the result's norm).
#define LX_NW 4
struct LxArgs {
  const bf16_t* q;           // [T][H][LX_D + DR]
  const bf16_t* kv;          // [rows][2][H][LX_D]: keys, values
  const bf16_t* rot;         // [rows][DR]
  bf16_t* out;               // [T][H][LX_D]
  const int* positions;
  const int* wi_seq;
  const int* wi_row0;
  const int* wi_count;
  const int* seq_start;
  const int* ctx_len;
  int n_items, H, first_round;
  float scale_log2e;
  const float* sink;         // [H] or null
  const bf16_t* gate;
  int gate_ld, gate_col, gate_mode;      // 0: none; 1: a number a head; 2: a number an element
};

template <int DR>
__global__ void __launch_bounds__(LX_NW * 64, 2)
latent_expanded_kernel(LxArgs a) {
  static_assert(DR == 0 || DR == 64, "a key's rotated part has eight pieces");
  constexpr int NW = LX_NW, DK = LX_D + DR;
  constexpr int KSTEPS = DK / 32, DBLK = LX_D / 16, JB = LX_KT / 16, KK = LX_KT / 32;
  constexpr int VB = LX_D * 2;                               // bytes of a value and of a key's first part
  constexpr int VALUES_AT = LX_KT * VB, ROT_AT = 2 * LX_KT * VB, PLACE = ROT_AT + LX_KT * DR * 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char lx_lds[];      // [2][keys, values, rotated parts]

  // the items with most keys first; those that start as second workgroups of a compute unit the other way round
  const int h = blockIdx.x, y = blockIdx.y;
  const int item = y < a.first_round ? a.n_items - 1 - y : y - a.first_round;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, grp = lane >> 4;
  const int seq = a.wi_seq[item], row0 = a.wi_row0[item], count = min(a.wi_count[item], LX_ROWS);
  if (count <= 0) return;
  // where the request's rows begin: behind all tokens and contexts before it
  int first = 0;
  for (int s = lane; s < seq; s += 64) first += a.ctx_len[s];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) first += __shfl_xor(first, o, ZA_WAVE);
  first = __builtin_amdgcn_readfirstlane(first + a.seq_start[seq]);
  const int hi = __builtin_amdgcn_readfirstlane(a.positions[row0 + count - 1]);

  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const int row = wave * 16 + r16, tok = row0 + (row < count ? row : 0);
  const int pos = row < count ? a.positions[tok] : -1;
  bf16x8_t qf[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(a.q + ((size_t)tok * a.H + h) * DK + ks * 32 + grp * 8);
    qf[ks] = row < count ? x : zero8;
  }
  // what the wave's rows see: all of them the keys up to wave_lo, some those up to wave_hi
  const bool wave_full = wave * 16 + 16 <= count;
  const int wave_hi = wave * 16 < count ? __builtin_amdgcn_readfirstlane(a.positions[row0 + min(wave * 16 + 16, count) - 1]) : -1;
  const int wave_lo = wave * 16 < count ? __builtin_amdgcn_readfirstlane(a.positions[row0 + wave * 16]) : 0;

  // ---- the requests for a tile: a wave brings 64 pieces of 16 bytes at a time, lane after lane (keys beyond the item's
  // last one read that one; their scores are masked)
  const unsigned kv_ld = 4u * a.H * LX_D;                    // bytes of a row
  const char* kv = (const char*)a.kv + (size_t)first * kv_ld + (size_t)h * VB;
  const char* rot = DR ? (const char*)a.rot + (size_t)first * (DR * 2) : nullptr;
  const unsigned lds = lds_address(lx_lds);
  auto bring = [&](const char* from, unsigned at, unsigned to) {
    asm volatile("s_mov_b32 m0, %0\n" "s_nop 0\n" "global_load_lds_dwordx4 %1, %2\n"
                 :: "s"(to), "v"(at), "s"(from) : "memory", "m0");
  };
  auto request = [&](int tile0, unsigned place) {
#pragma unroll
    for (int i = 0; i < LX_KT / 4 / NW; ++i) {
      const int key = (i * NW + wave) * 4 + grp;
      const unsigned at = (unsigned)min(tile0 + key, hi) * kv_ld, k7 = key & 7, to = place + (i * NW + wave) * 1024;
      bring(kv, at + ((r16 ^ k7) << 4), to);
      bring(kv + (size_t)a.H * VB, at + ((r16 ^ (k7 << 1)) << 4), to + VALUES_AT);
    }
    if constexpr (DR > 0)
#pragma unroll
      for (int i = 0; i < LX_KT / 8 / NW; ++i) {
        const int key = (i * NW + wave) * 8 + (lane >> 3);
        bring(rot, (unsigned)min(tile0 + key, hi) * (DR * 2) + (((lane & 7) ^ (key & 7)) << 4),
              place + ROT_AT + (i * NW + wave) * 1024);
      }
  };
  // all waves' requests have arrived, and the tile before them has been read
  auto arrived = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4_t o[DBLK], lsum = {0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY;
  bf16x8_t ones8;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones8[i] = (bf16_t)1.0f;
#pragma unroll
  for (int db = 0; db < DBLK; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // a lane's place in a fragment of keys; and in one of values: of the four keys that it points at (and the
  // four sixteen on) the lane's channels
  const int k_at = r16 * VB + ((grp ^ (r16 & 7)) << 4), rot_at = ROT_AT + r16 * DR * 2 + ((grp ^ (r16 & 7)) << 4);
  const int v_key = grp * 4 + (r16 >> 2);
  const int v_at = VALUES_AT + v_key * VB + ((((r16 >> 1) & 1) ^ ((v_key & 7) << 1)) << 4) + (r16 & 1) * 8;

  request(0, lds);
  arrived();
  const int n_tiles = hi / LX_KT + 1;
  for (int t = 0; t < n_tiles; ++t) {
    const int tile0 = t * LX_KT;
    const unsigned char* place = lx_lds + (t & 1) * PLACE;
    if (t + 1 < n_tiles) request(tile0 + LX_KT, lds + ((t + 1) & 1) * PLACE);
    if (tile0 <= wave_hi) {
      auto read_keys = [&](int ks, bf16x8_t (&f)[JB]) {
#pragma unroll
        for (int jb = 0; jb < JB; ++jb)
          f[jb] = *reinterpret_cast<const bf16x8_t*>(
              place + (ks < LX_D / 32 ? jb * 16 * VB + (k_at ^ ((ks & 1) << 6)) + (ks >> 1) * 128
                                      : jb * 16 * DR * 2 + (rot_at ^ ((ks & 1) << 6))));
      };
      auto read_values = [&](int group, bf16x8_t (&f)[4]) {      // 32 keys, four times 16 channels
        const int kk = group / (DBLK / 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int db = group % (DBLK / 4) * 4 + i;
          bf16x4_t half[2];
#pragma unroll
          for (int hf = 0; hf < 2; ++hf)
            half[hf] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
                (__attribute__((address_space(3))) bf16x4_t*)(place + (v_at ^ (db << 5)) + (kk * 32 + hf * 16) * VB));
          f[i] = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
        }
      };
      f32x4_t s[JB];
#pragma unroll
      for (int jb = 0; jb < JB; ++jb) s[jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      bf16x8_t kf[2][JB], vf[2][4];
      read_keys(0, kf[0]);
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        if (ks + 1 < KSTEPS) read_keys(ks + 1, kf[(ks + 1) & 1]);
        else read_values(0, vf[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int jb = 0; jb < JB; ++jb)
          s[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks & 1][jb], qf[ks], s[jb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // (a tile every key of which counts for every row of the wave needs no mask)
      if (!wave_full || tile0 + LX_KT - 1 > wave_lo) {
        const int last = pos - tile0 - grp * 4;
#pragma unroll
        for (int jb = 0; jb < JB; ++jb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (jb * 16 + i > last) s[jb][i] = -INFINITY;
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int jb = 0; jb < JB; ++jb)
#pragma unroll
        for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[jb][i]);
      tmax = quad_max(tmax);
      const float m_new = fmaxf(m, tmax * a.scale_log2e);      // (the factor is positive)
      const float m_use = m_new > -INFINITY ? m_new : 0.f;
      const float alpha = m == m_new || m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_use);
#pragma unroll
      for (int jb = 0; jb < JB; ++jb)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[jb][i] = __builtin_amdgcn_exp2f(fmaf(s[jb][i], a.scale_log2e, -m_use));
      m = m_new;
      if (__any(alpha != 1.0f)) {
        lsum *= alpha;
#pragma unroll
        for (int db = 0; db < DBLK; ++db) o[db] *= alpha;
      }
      bf16x8_t pf[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pf[kk][i] = (bf16_t)s[2 * kk][i];
          pf[kk][4 + i] = (bf16_t)s[2 * kk + 1][i];
        }
        // (the sum of the rounded probabilities)
        lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones8, pf[kk], lsum, 0, 0, 0);
      }
      constexpr int GROUPS = KK * (DBLK / 4);
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        if (g + 1 < GROUPS) read_values(g + 1, vf[(g + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        const int kk = g / (DBLK / 4), db0 = g % (DBLK / 4) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[db0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[g & 1][i], pf[kk], o[db0 + i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    arrived();
  }

  if (pos < 0) return;
  float total = lsum[0];
  if (a.sink && m > -INFINITY) total += exp2f(a.sink[h] * ZA_LOG2E - m);
  float inv = total > 0.f ? 1.0f / total : 0.f;
  const bf16_t* gate = a.gate_mode ? a.gate + (size_t)tok * a.gate_ld + a.gate_col : nullptr;
  if (a.gate_mode == 1) inv *= 1.0f / (1.0f + expf(-(float)gate[h]));
  bf16_t* to = a.out + ((size_t)tok * a.H + h) * LX_D + grp * 4;
#pragma unroll
  for (int db = 0; db < DBLK; ++db) {
    f32x4_t x = o[db] * inv;
    if (a.gate_mode == 2) {
      const bf16x4_t g = *reinterpret_cast<const bf16x4_t*>(gate + (size_t)h * LX_D + db * 16 + grp * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] *= 1.0f / (1.0f + expf(-(float)g[i]));
    }
    bf16x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (bf16_t)x[i];
    *reinterpret_cast<bf16x4_t*>(to + db * 16) = v;
  }
}

template <int DR>
static int launch_latent_expanded(const LxArgs& a, hipStream_t stream) {
  constexpr int LDS = 2 * LX_KT * (2 * LX_D + DR) * 2;
  auto kernel = latent_expanded_kernel<DR>;
  static bool allowed = false;
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  hipLaunchKernelGGL(kernel, dim3(a.H, a.n_items), dim3(LX_NW * 64), LDS, stream, a);
  return za_launch_status();
}

// Work items of at most LX_ROWS consecutive tokens of one request; `kv` and `rot` hold every request's visible rows, one
// request's behind the other's (ctx_len of them, then its tokens), n_rows in all or fewer.
extern "C" int za_latent_expanded(const void* q, const void* kv, const void* rot, int n_rows, void* out,
                                  const int* positions, const int* wi_seq, const int* wi_row0, const int* wi_count,
                                  const int* seq_start, const int* ctx_len, int n_items, int H, int Dr, float scale,
                                  const float* sink, const void* gate, int gate_ld, int gate_col, int gate_mode,
                                  hipStream_t stream) {
  if (n_items == 0) return 0;
  if (n_items < 0 || H <= 0 || n_rows <= 0 || !q || !kv || (Dr > 0 && !rot) || !out || !positions || !wi_seq ||
      !wi_row0 || !wi_count || !seq_start || !ctx_len || gate_mode < 0 || gate_mode > 2 ||
      (gate_mode && (!gate || gate_col < 0)))
    return ZA_ERR_ARG;
  // (a request's rows are reached by 32-bit offsets in bytes)
  if ((Dr != 0 && Dr != 64) || n_items > 65535 || (long long)n_rows * H * LX_D * 4 > 0xffffffffLL ||
      (gate_mode == 2 && (gate_ld % 4 || gate_col % 4 || (reinterpret_cast<uintptr_t>(gate) & 7))) ||
      ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kv) | reinterpret_cast<uintptr_t>(rot) |
        reinterpret_cast<uintptr_t>(out)) & 15))
    return ZA_ERR_UNSUPPORTED;
  // two workgroups a compute unit: where they all start at once, the second ones turned round even the chains out
  // (1,777 tokens 39.4 for 41.0; 4,096, which come in rounds, 126 for 116)
  const int first_round = (long long)n_items * H <= 512 ? min(256 / H, n_items) : n_items;
  const LxArgs a{(const bf16_t*)q, (const bf16_t*)kv, (const bf16_t*)rot, (bf16_t*)out, positions, wi_seq, wi_row0,
                 wi_count, seq_start, ctx_len, n_items, H, first_round, scale * ZA_LOG2E, sink, (const bf16_t*)gate,
                 gate_ld, gate_col, gate_mode};
  return Dr ? launch_latent_expanded<64>(a, stream) : launch_latent_expanded<0>(a, stream);
}
