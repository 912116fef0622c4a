// Float32 prompt attention over the paged cache for heads of 32, 64, 96 and 128 and pages of a multiple of 16 slots; formulas, operands and
// precision as in attention_f32.hip, whose kernel of 32 columns stays for other sizes, for many short chains of tiles and for decode tokens.
//
// A workgroup takes 32 consecutive tokens of one request and one head; its four waves take the tiles of 32 keys in turn and meet in LDS at the
// end.  (One wave to 32 tokens and all of their keys, as in the other kernel: at 700 tokens of 32 heads 704 waves on 1,024 SIMDs, the longest
// with 22 tiles in a row.)  A wave's tiles are its own: its keys and values go from the pages into its part of LDS without registers and
// without a barrier, each into the one place that the tile before has just been read from, the keys beside softmax and values, the values
// beside the scores.  What bounds it: a tile's 64 matrix instructions of heads of 64 are 4,096 cycles, and the vector instructions, which
// do not run beside them, came on top with 1,900 when the exponentials were expf; now 1,350.  (The next tile's scores between this one's
// exponentials: no faster for heads of 64, slower for 128.)  In a replayed graph, us, before and now: 32 heads of 64, 45 tokens 13.0 / 6.9, 200 30.7 /
// 10.1, 700 84 / 36, 2,048 234 / 177, 20 behind 1,000 117 / 26, four prompts of 500 73 / 68; 32 of 128, 700 134 / 66; errors against 64 bits
// 3.0e-7 / 2.5e-7 at 700 tokens.
#pragma once
#include <math.h>

#include "common.hpp"

namespace kllm {

template <int HDT>
struct F32PromptShape {
  static constexpr int hd = 32 * HDT;
  static constexpr int CH = hd / 4;                 // 16-byte pieces of a key's row
  static constexpr int TB = 32 * hd * 4;            // bytes of a tile's keys, and of its values
  static constexpr int DI = TB / 1024;              // load instructions for either, half of them for each 16 keys
};

template <int HDT>   // head_dim = 32 * HDT
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn_f32_prompt_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ cache, const int* __restrict__ query_tiles, int n_tiles,
    const int* __restrict__ span_start, const int* __restrict__ span_pos, const int* __restrict__ block_table, int max_pages, int page_size,
    int H, int KV, int window, int chunk, const float* __restrict__ sinks, float scale, const float* __restrict__ slopes, const OutGate gate) {
  typedef F32PromptShape<HDT> S;
  constexpr int hd = S::hd, CH = S::CH, TB = S::TB, DI = S::DI, KC = hd / 8;
  extern __shared__ __attribute__((aligned(1024))) unsigned char f32_lds[];   // [wave][keys, values][TB]
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 32, c = lane % 32;
  // Longest first; neighbouring heads, which share keys, on one XCD.
  const int place = (int)(blockIdx.x / H), pair = 4 * n_tiles - 1 - place;
  int h = (int)(blockIdx.x % H);
  if (H % 8 == 0) h = h % 8 * (H / 8) + h / 8;
  const int blk = pair / 4, sub = pair % 4, kvh = h / (H / KV);
  const int t0 = __builtin_amdgcn_readfirstlane(query_tiles[2 * blk]) + 32 * sub;
  const int span = __builtin_amdgcn_readfirstlane(query_tiles[2 * blk + 1]);
  const int s_begin = __builtin_amdgcn_readfirstlane(span_start[span]), s_end = __builtin_amdgcn_readfirstlane(span_start[span + 1]);
  if (t0 >= s_end) return;                                    // the block ends before these 32 tokens: the whole workgroup
  const int ncol = min(32, s_end - t0);
  const int pos_base = __builtin_amdgcn_readfirstlane(span_pos[span]) + (t0 - s_begin);
  const int cc = min(c, ncol - 1), my_pos = pos_base + cc, tok = t0 + cc;
  const int my_start = first_key(my_pos, window, chunk);
  const int qmax = pos_base + ncol - 1;                       // last key any column reads
  const int lowest = first_key(pos_base, window, chunk);      // first key any column reads
  const int highest_start = first_key(qmax, window, chunk);   // from here on no column masks a key below it
  const int first = lowest / 32 * 32;
  const int tiles = (qmax - first) / 32 + 1;
  const int first_page_key = lowest / page_size * page_size;  // pages before this may be gone
  const float my_slope = slopes ? slopes[h] : 0.f;

  floatx4 qb[KC];                                             // this column's query, floats 8 kk + 4 g ...
#pragma unroll
  for (int kk = 0; kk < KC; ++kk) qb[kk] = *reinterpret_cast<const floatx4*>(q + ((long)tok * H + h) * hd + 8 * kk + 4 * g);

  // ---- where the wave's t-th tile (4 t + wave) is: lane i has half i % 2 (16 keys, in one page) of the tile first_t + i / 2
  const int* table = block_table + (long)span * max_pages;
  const long block = (long)page_size * hd;
  const unsigned page_bytes = (unsigned)(2 * KV * block * 4);
  const unsigned k_head = (unsigned)(kvh * block * 4), v_head = (unsigned)((KV + kvh) * block * 4);
  unsigned at_lo, at_hi, at_v;
  auto lookup = [&](int first_t) __attribute__((always_inline)) {
    const int key0 = first + 32 * (4 * (first_t + lane / 2) + wave) + 16 * (lane % 2);
    const bool ok = (key0 <= qmax) & (key0 + 15 >= first_page_key);
    const int index = key0 / page_size;
    const unsigned slot0 = (unsigned)(key0 - index * page_size), page = (unsigned)max(table[ok ? index : 0], 0);
    const unsigned long at = reinterpret_cast<unsigned long>(cache) + (unsigned long)page * page_bytes + (k_head + slot0 * (unsigned)(hd * 4));
    at_lo = (unsigned)at;
    at_hi = (unsigned)(at >> 32);
    at_v = (v_head - k_head) - slot0 * (unsigned)(hd * 4 - 4);
  };
  // Lane l's 16 bytes land at base + 16 l, so lanes choose what they fetch: a key's row keeps its pieces, and a column's four of 16 keys
  // theirs, exchanged so that a read of 16 rows meets all banks.
  auto ksw = [](int row) { return CH % 16 == 0 ? row & 15 : (row >> 1) & 7; };
  unsigned koff[DI / 2], voff;
#pragma unroll
  for (int i = 0; i < DI / 2; ++i) {
    const int piece = 64 * i + lane, row = piece / CH;
    koff[i] = (unsigned)(row * hd * 4 + ((piece % CH) ^ ksw(row)) * 16);
  }
  voff = (unsigned)((lane / 4) * page_size + ((lane % 4) ^ ((lane >> 4) & 3)) * 4) * 4u;
  unsigned char* const kt = f32_lds + wave * (2 * TB);
  unsigned char* const vt = kt + TB;
  auto dma = [&](const char* src, unsigned off, unsigned char* dst) {
    asm volatile("" : "+v"(off));                             // (or the loop keeps 64-bit offsets)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off),
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };
  auto place_of = [&](int t, int half) {
    const int i = 2 * (t % 32) + half;
    const unsigned lo = __builtin_amdgcn_readlane(at_lo, i), hi = __builtin_amdgcn_readlane(at_hi, i);
    return reinterpret_cast<const char*>((unsigned long)hi << 32 | lo);
  };
  auto load_k = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const char* src = place_of(t, half);
#pragma unroll
      for (int i = 0; i < DI / 2; ++i) dma(src, koff[i], kt + (half * (DI / 2) + i) * 1024);
    }
  };
  auto load_v = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const char* src = place_of(t, half) + (int)__builtin_amdgcn_readlane(at_v, 2 * (t % 32) + half);
#pragma unroll
      for (int i = 0; i < DI / 2; ++i) dma(src + (long)(16 * i) * page_size * 4, voff, vt + (half * (DI / 2) + i) * 1024);
    }
  };
  auto fence = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
#define KLLM_VM_WAIT(VM) __builtin_amdgcn_s_waitcnt(((VM) & 0xF) | (((VM) >> 4) << 14) | 0x0F70)

  const int kat = c * (CH * 16) + ((g ^ (ksw(c) & 1)) * 16);  // piece 2 kk + g: kat ^ 32 (kk ^ half of the row's exchange)
  const int kx = (ksw(c) & ~1) * 16;
  float m = -INFINITY, l = 0.f;
  if (sinks && wave == 0) {                                   // a key with a score of its own and no value; one of a column's lanes has its term
    m = sinks[h];
    l = g == 0 ? 1.f : 0.f;
  }
  const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  floatx16 acc[HDT];
#pragma unroll
  for (int r = 0; r < HDT; ++r) acc[r] = zero16;

  const int mine = (tiles - wave + 3) / 4;                    // tiles of this wave
  if (mine > 0) {
    lookup(0);
    load_k(0);
    load_v(0);
  }
  for (int t = 0; t < mine; ++t) {
    const int kb = first + 32 * (4 * t + wave);
    const bool more = t + 1 < mine;
    // ---- scores
    fence();
    KLLM_VM_WAIT(DI);                                         // the keys have landed; the values may be on their way
    fence();
    floatx16 s = zero16;
#pragma unroll
    for (int kk = 0; kk < KC; ++kk) {
      const floatx4 a = *reinterpret_cast<const floatx4*>(kt + (kat + (kx ^ (32 * kk))));
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], qb[kk][e], s, 0, 0, 0);
    }
    fence();
    __builtin_amdgcn_s_waitcnt(0xC07F);                       // (the last keys are read: their place takes the next tile's)
    if (more) {
      if ((t + 1) % 32 == 0) {                                // (the values of this tile are asked for already)
        lookup(t + 1);
      }
      load_k(t + 1);
    }
    fence();
    // ---- mask, running maximum and sum; s becomes the probabilities.  (The scale by itself: in one instruction with the subtraction of the maximum,
    // which was rounded, the largest scores would be off from it by half of its last place, which is more than exponentials bear from 2^31 on.)
    if (slopes) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], scale, -my_slope * (float)(my_pos - (kb + 8 * (i / 4) + 4 * g + i % 4)));
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] *= scale;
    }
    if ((kb < highest_start) | (kb + 31 > pos_base)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = kb + 8 * (i / 4) + 4 * g + i % 4;
        s[i] = (key <= my_pos) & (key >= my_start) ? s[i] : -INFINITY;
      }
    }
    float tmax = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
    const unsigned w = __builtin_bit_cast(unsigned, tmax);
    const auto x = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    tmax = fmaxf(__builtin_bit_cast(float, (unsigned)x[0]), __builtin_bit_cast(float, (unsigned)x[1]));
    if (__any(tmax > m)) {                                    // (otherwise everything is multiplied by one)
      const float m_new = fmaxf(m, tmax);
      const float alpha = exp_negative(m - (m_new == -INFINITY ? 0.f : m_new));
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int r = 0; r < HDT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][i] *= alpha;
    }
    const float mref = (m == -INFINITY) ? 0.f : m;            // a column with no key yet
    float psum = 0.f;
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] = exp_negative(s[i] - mref);
        psum += s[i];
      }
    }
    l += psum;
    // ---- values
    fence();
    if (more) KLLM_VM_WAIT(DI);                               // the values have landed; the next keys may be on their way
    else KLLM_VM_WAIT(0);
    fence();
    if ((kb < first_page_key) | (kb + 31 > qmax)) {           // slots that may hold anything
#pragma unroll
      for (int i = 0; i < DI; ++i) {
        floatx4* at = reinterpret_cast<floatx4*>(vt + 1024 * i + 16 * lane);
        const int key = kb + 16 * (i / (DI / 2)) + 4 * ((lane % 4) ^ ((lane >> 4) & 3));
        floatx4 v = *at;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (key + e >= first_page_key) & (key + e <= qmax) ? v[e] : 0.f;
        *at = v;
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);
      fence();
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < HDT; ++r) {
        const int piece = (2 * j + g) % 4;                    // of the half j / 2
        const floatx4 v = *reinterpret_cast<const floatx4*>(vt + (j / 2) * (hd * 64) + (32 * r + c) * 64 + (piece ^ ((c >> 2) & 3)) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[r] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], s[4 * j + e], acc[r], 0, 0, 0);
      }
    fence();
    __builtin_amdgcn_s_waitcnt(0xC07F);
    if (more) load_v(t + 1);
  }
#undef KLLM_VM_WAIT
  l += __shfl_xor(l, 32, kWave);

  // ---- the waves meet: each leaves its sums in its part of LDS, lane-contiguous, and writes a quarter of the output's rows
  float* const red = reinterpret_cast<float*>(kt);
#pragma unroll
  for (int r = 0; r < HDT; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      *reinterpret_cast<floatx4*>(red + ((r * 4 + b) * kWave + lane) * 4) = floatx4{acc[r][4 * b], acc[r][4 * b + 1], acc[r][4 * b + 2], acc[r][4 * b + 3]};
  float* const ml = red + HDT * 16 * kWave;
  ml[lane] = m;                                               // -inf and 0 for a wave without a key for this column
  ml[kWave + lane] = l;
  __syncthreads();
  if (c >= ncol) return;
  float mw[4], M = -INFINITY, L = 0.f;
  const float* const all = reinterpret_cast<const float*>(f32_lds);
  constexpr int kPart = 2 * TB / 4;                           // floats of a wave's part
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    mw[w] = all[w * kPart + HDT * 16 * kWave + lane];
    M = fmaxf(M, mw[w]);
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    mw[w] = exp_negative(mw[w] - M);                          // (M is finite: a column reads its own key)
    L += mw[w] * all[w * kPart + HDT * 16 * kWave + kWave + lane];
  }
  const float inv = 1.f / L;
  float* const orow = out + ((long)tok * H + h) * hd;
#pragma unroll
  for (int r = 0; r < HDT; ++r) {
    const int d = 32 * r + 8 * wave + 4 * g;
    floatx4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(all + w * kPart + ((r * 4 + wave) * kWave + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += mw[w] * v[e];
    }
    const floatx4 og = out_gate4(gate, tok, h, d);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = o[e] * inv * og[e];
    *reinterpret_cast<floatx4*>(orow + d) = o;
  }
}

}  // namespace kllm
