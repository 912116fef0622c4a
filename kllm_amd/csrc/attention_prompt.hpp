// Prompt attention over the paged cache (bfloat16), the kernel for heads of 32, 64 and 128 without a distance bias; the arithmetic of
// attn_prefill_mfma_kernel (attention_prefill.hip), which stays for the others.
//
// A workgroup takes up to 128 consecutive tokens of one request and one head, a wave of a group of four 32 of them; with PAR = 2 two groups
// take the tiles of keys in turn and meet in LDS at the end.  What bounds it is instructions: the matrix products of 32 queries and 64
// keys of 64 take 640 cycles, exponentials, maximum and conversions 600, and whatever else a tile costs comes on top (before: 265 vector
// and 166 scalar instructions a wave and tile, of which 100 are the arithmetic; now 149 and 50).  So
// - tiles go from the pages into LDS without registers (16 bytes a lane, three tiles in a ring).  A wave moves 16 keys (8 of heads of 128)
//   and the values of 16, which lie in one page: it has one address a tile, worked out for 64 tiles at a time, a tile to a lane.
// - LDS holds no padding; keys lie in their rows' pieces exchanged, values [16 keys][head column] as in the pages with their two pieces
//   exchanged in every other eight columns: every read is 16 bytes a lane without a bank conflict.
// - A's row r is key (r's bits 2 and 3 exchanged), so that the eight scores a lane has of sixteen keys belong to eight neighbouring ones,
//   whose values are one read (two of 8 bytes before).
// - the sum of the probabilities is an accumulator like the output's; a branch around matrix products makes the compiler copy
//   accumulators, so values of keys that do not exist become zeros in LDS, and there is one copy of the products.
// - the exponentials of sixteen keys stand beside the products of the sixteen before, and the next tile's loads behind the scores' products.
// In a replayed graph, us, before and now: 32 heads of 64, 2,048 tokens 47 / 35, 700 18.4 / 12.3, 500 behind 1,000 28 / 21, 8,192 431 / 345; 32 of
// 128, 2,048 73 / 52, three prompts of 1,999 together 46 / 32, 480 behind 480 31 / 21, 20 behind 500 21.6 / 13.5, 45 11.3 / 6.6.  Tried and not kept:
// the scores of the next tile beside this one's exponentials, with a second set of accumulators (registers: the sets go through scratch memory).
#pragma once
#include <math.h>

#include <type_traits>

#include "common.hpp"

namespace kllm {

constexpr int kPrefillMaxPage = 2048;             // limits of the division-free page arithmetic (page_magic)
constexpr int kPrefillMaxKeys = 1 << 24;
constexpr int kPrefillSliceFromKeys = 1280;       // the keys of a block go in slices when the longest block reads at least this many

template <int HDT>
struct PromptShape {
  static constexpr int hd = 32 * HDT;
  static constexpr int KS = hd / 16;
  static constexpr int NB = HDT <= 2 ? 2 : 1;       // blocks of 32 keys in a tile
  static constexpr int KT = 32 * NB;                // keys of a tile
  static constexpr int CH = 4 * HDT;                // 16-byte pieces of a key's row
  static constexpr int TB = KT * hd * 2;            // bytes of a tile's keys, and of its values
  static constexpr int DI = TB / 4096;              // load instructions of a wave for either
  static constexpr int RING = 3;                    // tiles in LDS
};

template <int HDT, int PAR>  // head_dim = 32 * HDT; PAR groups of four waves
__device__ __forceinline__ void attn_prompt_block(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
    const int* __restrict__ query_tiles, int n_tiles, const int* __restrict__ span_start,
    const int* __restrict__ span_pos, const int* __restrict__ block_table, int max_pages,
    int page_size, unsigned page_magic, int H, int KV, int window, int chunk, const float* __restrict__ sinks, int keep_first,
    float scale, float* __restrict__ part, const OutGate gate, int place, int slice, int nslices) {
  typedef PromptShape<HDT> S;
  constexpr int hd = S::hd, KS = S::KS, NB = S::NB, KT = S::KT, CH = S::CH, TB = S::TB, DI = S::DI, RING = S::RING;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring_lds[];   // [PAR][RING][keys, values][TB]
  const int lane = threadIdx.x % kWave;
  const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int par = wave8 / 4, wave = wave8 % 4;               // the group: tiles par, par + PAR, ...
  const int g = lane / 32, c = lane % 32;
  const int item = place;                                // (block, head), head fastest
  // Later blocks read more keys.  With several workgroups a CU (one group) the later half of the list starts first, longest block first, then
  // the earlier half, shortest first, so that a CU gets a long and a short one; with one workgroup a CU longest first throughout.
  const int turn = item / H, n_late = (n_tiles + 1) / 2;
  int h = item % H;
  if (H % 8 == 0) h = h % 8 * (H / 8) + h / 8;               // neighbouring heads, which share keys, on one XCD
  const int blk = (PAR == 2 || turn < n_late) ? n_tiles - 1 - turn : turn - n_late;
  const int kvh = h / (H / KV);
  const int t0 = __builtin_amdgcn_readfirstlane(query_tiles[2 * blk]);
  const int span = __builtin_amdgcn_readfirstlane(query_tiles[2 * blk + 1]);
  const int s_begin = __builtin_amdgcn_readfirstlane(span_start[span]);
  const int s_end = __builtin_amdgcn_readfirstlane(span_start[span + 1]);
  const int pos0 = __builtin_amdgcn_readfirstlane(span_pos[span]);
  const int kv_len = pos0 + (s_end - s_begin);              // keys of the request after this step
  const int nq_blk = min(128, s_end - t0);
  const int blk_qmin = pos0 + (t0 - s_begin), blk_qmax = blk_qmin + nq_blk - 1;
  const int wq0 = t0 + 32 * wave;
  const int nq = max(0, min(32, s_end - wq0));
  const bool active = nq > 0;
  const int tq = active ? wq0 + min(c, nq - 1) : t0;        // this lane's query (clamped)
  const int qpos = pos0 + (tq - s_begin);
  const int w_qmin = pos0 + (wq0 - s_begin), w_qmax = w_qmin + nq - 1;
  const int lowest = first_key(blk_qmin, window, chunk);      // first key any query reads
  const int w_highstart = first_key(w_qmax, window, chunk);   // from here on no query of the wave masks a key below it
  const int my_start = first_key(qpos, window, chunk);
  const int* table = block_table + (long)span * max_pages;
  const float c2 = scale * 1.4426950408889634f;             // scale * log2(e)

  bf16x8 qb[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
    qb[kk] = *reinterpret_cast<const bf16x8*>(q + ((long)tq * H + h) * hd + 16 * kk + 8 * g);

  // Kept first positions: the keys below kept_end (none of them in the tiles from kb0 on) come first, in n_kept tiles of their own from key
  // 0; pages between them and kb0 may be gone.  The tiles go in turn to the slices and, within a slice, to the groups.
  const int kb0 = lowest / 32 * 32;
  const int kept_end = min(keep_first, kb0);
  const int n_kept = (kept_end + KT - 1) / KT;
  const int ntiles_all = (blk_qmax - kb0) / KT + 1 + n_kept;
  const int ntiles = (ntiles_all + PAR * nslices - 1) / (PAR * nslices);   // steps of the loop: the same for all
  auto tile_no = [&](int t) { return nslices * (PAR * t + par) + slice; };
  auto first_of = [&](int n) { return n < n_kept ? KT * n : kb0 + KT * (n - n_kept); };   // first key of a tile
  // Page of a key without a division: page_magic = ceil(2^35 / page_size), exact for keys below 2^24 and pages of up to 2,048 tokens.
  auto page_index = [&](int key) { return (int)(__umulhi((unsigned)key, page_magic) >> 3); };
  const int first_page_key = page_index(lowest) * page_size;   // pages before this may be gone
  // Tiles up to read_end hold keys for this wave; from bulk_begin to bulk_end every key is for all of its queries; from whole_begin to
  // whole_end every key exists, and so does its page.
  const int read_end = active ? n_kept + (w_qmax - kb0) / KT + 1 : 0;
  const int bulk_begin = n_kept + (max(w_highstart - kb0, 0) + KT - 1) / KT, bulk_end = n_kept + (w_qmin + 1 - kb0) / KT;
  const int whole_begin = n_kept + (kb0 < first_page_key), whole_end = n_kept + (kv_len - kb0) / KT;
  auto key_ok = [&](int key) { return (key < kv_len) & ((key >= first_page_key) | (key < keep_first)); };

  // ---- a tile's way into LDS: lane l's 16 bytes land at base + 16 l, so lanes choose what they fetch.  A half (16 keys) lies in one page; one
  // that does not exist reads page 0 and is masked (keys) or cleared (values).
  const long block = (long)page_size * hd;
  const unsigned page_bytes = (unsigned)(2 * KV * block * 2);
  const unsigned k_head = (unsigned)(kvh * block * 2), v_head = (unsigned)((KV + kvh) * block * 2);
  const int my_half = wave * DI * (64 / CH) / 16;             // of the tile's 16 keys each
  unsigned koff[DI], voff[DI];
#pragma unroll
  for (int i = 0; i < DI; ++i) {
    const int row = (wave * DI + i) * (64 / CH) + lane / CH;
    const int sw = CH == 8 ? (row >> 1) & 7 : CH == 16 ? row & 15 : (row >> 2) & 3;
    koff[i] = (unsigned)((row % 16) * hd + ((lane % CH) ^ sw) * 8) * 2u;
    const int d = ((wave * DI + i) % HDT) * 32 + lane / 2;
    voff[i] = (unsigned)(d * page_size + ((lane % 2) ^ ((lane >> 4) & 1)) * 8) * 2u;
  }
  unsigned char* const ring = ring_lds + par * (2 * RING * TB);
  // Lane i: where this wave's half of tile first + i begins, its keys' first row (64 bits) and from there its values' first slot.
  const char* const cache_bytes = reinterpret_cast<const char*>(cache);
  unsigned at_lo, at_hi, at_v;
  auto lookup = [&](int first) __attribute__((always_inline)) {
    const int t = first + lane;
    const int key0 = first_of(tile_no(t)) + 16 * my_half;
    const bool ok = (tile_no(t) < ntiles_all) & key_ok(key0);
    const int index = page_index(key0);
    const unsigned slot0 = (unsigned)(key0 - index * page_size), page = (unsigned)max(table[ok ? index : 0], 0);
    const unsigned long at = reinterpret_cast<unsigned long>(cache_bytes) + (unsigned long)page * page_bytes + (k_head + slot0 * (unsigned)(hd * 2));
    at_lo = (unsigned)at;
    at_hi = (unsigned)(at >> 32);
    at_v = (v_head - k_head) - slot0 * (unsigned)(hd * 2 - 2);
  };
  auto dma = [&](const char* src, unsigned off, unsigned char* dst) {
    asm volatile("" : "+v"(off));                             // (or the loop keeps 64-bit offsets)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off),
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };
  auto load = [&](int t, int slot) __attribute__((always_inline)) {
    const int i = t % 64;
    const unsigned lo = __builtin_amdgcn_readlane(at_lo, i), hi = __builtin_amdgcn_readlane(at_hi, i), dv = __builtin_amdgcn_readlane(at_v, i);
    const char* const k = reinterpret_cast<const char*>((unsigned long)hi << 32 | lo);
    const char* const v = k + (int)dv;
#pragma unroll
    for (int i = 0; i < DI; ++i) dma(k, koff[i], ring + slot * (2 * TB) + (wave * DI + i) * 1024);
#pragma unroll
    for (int i = 0; i < DI; ++i) dma(v, voff[i], ring + slot * (2 * TB) + TB + (wave * DI + i) * 1024);
  };
  auto fence = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto barrier = [&] {
    fence();
    __builtin_amdgcn_s_barrier();
    fence();
  };
#define KLLM_VM_WAIT(VM) __builtin_amdgcn_s_waitcnt(((VM) & 0xF) | (((VM) >> 4) << 14) | 0x0F70)

  // ---- operands
  const int krow = (c & 19) | ((c & 4) << 1) | ((c & 8) >> 1);
  const int ksw = CH == 8 ? (krow >> 1) & 7 : CH == 16 ? krow & 15 : (krow >> 2) & 3;
  const int kat = krow * (CH * 16) + ((g ^ ksw) * 16);
  const int vat = c * 32 + ((g ^ ((c >> 3) & 1)) * 16);
  constexpr float kGrow = 8.f;
  const bf16_t one = (bf16_t)1.f;
  bf16x8 ones = {one, one, one, one, one, one, one, one};
  asm volatile("" : "+v"(ones));
  const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  floatx16 acc[HDT], ls = zero16;
#pragma unroll
  for (int r = 0; r < HDT; ++r) acc[r] = zero16;
  const float grow_raw = kGrow / c2;                        // kGrow in units of raw scores
  float m = -INFINITY, mc = 0.f, m_limit = -INFINITY;       // maximum, m * c2 (0 while m is -inf), m + grow_raw
  if (sinks && par == 0 && slice == 0) {   // a key with a score of its own and no value
    m = sinks[h] / scale;
#pragma unroll
    for (int i = 0; i < 16; ++i) ls[i] = 1.f;
    mc = m * c2;
    m_limit = m + grow_raw;
  }

  constexpr int HALVES = 2 * NB;                            // of a tile: 16 keys each
  auto step = [&](int t, int n, int slot) __attribute__((always_inline)) {
    const unsigned char* const kt = ring + slot * (2 * TB);
    const unsigned char* const vt = kt + TB + vat;
    floatx16 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(kt + (kat ^ (32 * kk)) + b * (32 * CH * 16));
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qb[kk], kk == 0 ? zero16 : s[b], 0, 0, 0);
      }
    bf16x8 vf[2][HDT];                                        // the values of two halves of the tile
    auto read = [&](int x) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < HDT; ++r) vf[x % 2][r] = *reinterpret_cast<const bf16x8*>(vt + x * (hd * 32) + r * 1024);
    };
    read(0);
    read(1);
    fence();
    load(t + 2, slot == 0 ? 2 : slot - 1);                    // beside the products: its place among the instructions costs nothing here
    fence();
    if ((n < bulk_begin) | (n >= bulk_end)) {                 // some key is not for some query
      const bool kept_tile = n < n_kept;
      const int kb = first_of(n);
      const int hi = min(qpos, kv_len - 1) - kb - 8 * g;
      const int lo = kept_tile ? KT : my_start - kb - 8 * g;
      const int kf = (kept_tile ? kept_end : keep_first) - kb - 8 * g;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int e = 32 * b + 16 * (i / 8) + i % 8;
          const bool ok = (e <= hi) & ((e >= lo) | (e < kf));
          s[b][i] = ok ? s[b][i] : -INFINITY;
        }
    }
    float tmax = s[0][0];
#pragma unroll
    for (int e = 1; e < 16 * NB; ++e) tmax = fmaxf(tmax, s[e / 16][e % 16]);
    const unsigned w = __builtin_bit_cast(unsigned, tmax);
    const auto x = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    tmax = fmaxf(__builtin_bit_cast(float, (unsigned)x[0]), __builtin_bit_cast(float, (unsigned)x[1]));
    const bool grow = tmax > m_limit;                         // never for a maximum of -inf
    if (__any(grow)) {
      const float m_new = grow ? tmax : m;
      const float alpha = grow ? __builtin_amdgcn_exp2f(mc - m_new * c2) : 1.f;   // m = -inf: what was accumulated is 0 anyway
      const float a0 = (m == -INFINITY) ? 0.f : alpha;
      m = m_new;
      mc = (m == -INFINITY) ? 0.f : m * c2;
      m_limit = m + grow_raw;
#pragma unroll
      for (int i = 0; i < 16; ++i) ls[i] *= a0;
#pragma unroll
      for (int r = 0; r < HDT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][i] *= a0;
    }
    bf16x8 p[2];
    auto exponentials = [&](int x) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        p[x % 2][i] = (bf16_t)__builtin_amdgcn_exp2f(fmaf(s[x / 2][8 * (x % 2) + i], c2, -mc));   // exp2(-inf) = 0
    };
    exponentials(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < HALVES; ++x) {                        // a half's products beside the next one's exponentials
      ls = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, p[x % 2], ls, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < HDT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x % 2][r], p[x % 2], acc[r], 0, 0, 0);
      if (x + 1 < HALVES) exponentials(x + 1);
      if (x + 2 < HALVES) read(x + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Slots that may hold anything: this wave's values of keys that do not exist become zeros, before the barrier.
  auto clear = [&](int kb, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < DI; ++i) {
      bf16x8* at = reinterpret_cast<bf16x8*>(ring + slot * (2 * TB) + TB + (wave * DI + i) * 1024 + lane * 16);
      const int key = kb + 16 * my_half + ((lane % 2) ^ ((lane >> 4) & 1)) * 8;
      bf16x8 v = *at;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = key_ok(key + e) ? v[e] : (bf16_t)0.f;
      *at = v;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
  };

  // ---- the loop: tile t + 2 is asked for while t is multiplied; its page, two steps before
  lookup(0);
  load(0, 0);
  load(1, 1);
  int slot = 0;                                               // t % RING
  for (int t = 0; t < ntiles; ++t) {
    const int n = tile_no(t);
    KLLM_VM_WAIT(2 * DI);                                     // tile t has landed; in every wave, behind the barrier
    if ((n < whole_begin) | (n >= whole_end)) clear(first_of(n), slot);
    barrier();
    if ((t + 2) % 64 == 0) lookup(t + 2);
    if (n < read_end) step(t, n, slot);
    else load(t + 2, slot == 0 ? 2 : slot - 1);
    slot = slot == 2 ? 0 : slot + 1;
  }
  KLLM_VM_WAIT(0);
  float l = ls[0];

  // ---- the two groups meet: the second leaves maximum, sum and output in LDS (lane-contiguous), the first adds them with
  // weights exp(m - max m) and writes.
  if (PAR == 2) {
    float* red = reinterpret_cast<float*>(ring_lds);           // [4 waves][HDT*16 + 2][64]
    constexpr int kRows = HDT * 16 + 2;
    __syncthreads();                                           // the last tiles have been read
    float* mine = red + (wave * kRows) * kWave + lane;
    if (par == 1) {
#pragma unroll
      for (int r = 0; r < HDT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) mine[(16 * r + i) * kWave] = acc[r][i];
      mine[(HDT * 16) * kWave] = m;
      mine[(HDT * 16 + 1) * kWave] = l;
    }
    __syncthreads();
    if (par == 1) return;
    const float m1 = mine[(HDT * 16) * kWave], l1 = mine[(HDT * 16 + 1) * kWave];
    const float M = fmaxf(m, m1);
    // (M is -inf where neither group had a key for the lane's query: a slice of the keys that ends before it)
    const float w0 = (M == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m - M) * c2);   // exp2(-inf) = 0
    const float w1 = (M == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m1 - M) * c2);
    l = l * w0 + l1 * w1;
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][i] = acc[r][i] * w0 + mine[(16 * r + i) * kWave] * w1;
    m = M;
  }
  if (!active || c >= nq) return;
  if (nslices > 1) {
    // Keys in slices: the slice's sums as they are, with its maximum (in units of the scaled scores, as the merge takes it) and its
    // sum of probabilities; a slice without a key for this query leaves a maximum of -inf.  Rows of hd + 2 floats are 8-byte aligned.
    float* prow = part + (((long)tq * H + h) * nslices + slice) * (hd + 2);
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float* dst = prow + 32 * r + 8 * b + 4 * g;
        *reinterpret_cast<floatx2*>(dst) = floatx2{acc[r][4 * b], acc[r][4 * b + 1]};
        *reinterpret_cast<floatx2*>(dst + 2) = floatx2{acc[r][4 * b + 2], acc[r][4 * b + 3]};
      }
    if (g == 0) *reinterpret_cast<floatx2*>(prow + hd) = floatx2{m * scale, l};
    return;
  }
  const float inv = 1.f / l;                                  // finite: a query reads its own key
  bf16_t* orow = out + rows_at(gate.side, tq, h * hd + 4 * g, H * hd);
  auto store = [&](auto side) {                               // (eights of columns lie side times as far apart)
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const floatx4 og = out_gate4(gate, tq, h, 32 * r + 8 * b + 4 * g);
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16_t)(acc[r][4 * b + j] * inv * og[j]);
        *reinterpret_cast<bf16x4*>(orow + (32 * r + 8 * b) * side) = v;
      }
  };
  if (gate.side) store(gate.side);
  else store(std::integral_constant<int, 1>());
#undef KLLM_VM_WAIT
}

template <int HDT, int PAR>
__global__ __launch_bounds__(256 * PAR) __attribute__((amdgpu_waves_per_eu(PAR == 1 && HDT <= 2 ? 3 : 2))) void attn_prompt_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
    const int* __restrict__ query_tiles, int n_tiles, const int* __restrict__ span_start,
    const int* __restrict__ span_pos, const int* __restrict__ block_table, int max_pages,
    int page_size, unsigned page_magic, int H, int KV, int window, int chunk, const float* __restrict__ sinks, int keep_first,
    float scale, float* __restrict__ part, const OutGate gate) {
  attn_prompt_block<HDT, PAR>(q, out, cache, query_tiles, n_tiles, span_start, span_pos, block_table, max_pages, page_size, page_magic, H, KV, window,
                              chunk, sinks, keep_first, scale, part, gate, blockIdx.x, blockIdx.y, gridDim.y);
}

// Groups of four waves to a block of attn_prompt_kernel.  One group: a CU holds up to three blocks, and the longest block's chain of tiles, or
// the CU's share of all of them, follows on what a workgroup costs beside its tiles.  Two groups: a CU holds one block at a time, each with that
// cost, but a chain is half as long.  In us, per 64 keys.  (One group / two, measured: heads of 64, 2,048 tokens of 32 heads 37 / 35, 1,500
// 28 / 24, four prompts of 300 10.9 / 15.5, 17 blocks of three prompts 22 / 26, 8,192 tokens 341 / 342, 45 tokens 5.4 / 6.2; heads of 128, 2,048 59 / 51,
// three prompts 32 / 35, 480 behind 480 27 / 21, four prompts of 300 16 / 22.)
inline int prompt_groups(int hdt, int grid, int H, long keys_total, int keys_longest) {
  const int cus = device_cus();
  if (keys_total <= 0 || keys_longest <= 0) return grid > 2 * cus ? 1 : 2;      // not known
  const float longest = keys_longest / 64.f, share = (float)keys_total * H / (64.f * cus);
  const bool wide = hdt > 2;
  const float one = 5.f + fmaxf(longest * (wide ? 1.45f : 0.85f), share * (wide ? 1.1f : 0.65f));
  const float two = 1.5f + 4.5f * ceil_div(grid, cus) + fmaxf(longest, share) * (wide ? 1.1f : 0.6f);
  return two < one ? 2 : 1;
}

}  // namespace kllm
