// Float32 attention over the paged cache on the matrix cores, for prompts and
// for decode tokens: one kernel, two ways of filling its 32 columns, and behind it one of 16 columns
// that most decode tokens run on.
//
// Operands, products and sums are 32-bit throughout (MFMA 32x32x2 with float32
// inputs; expf; no reduced precision anywhere).  Formulas as in the generic
// kernel (reference: backend/model.cu:343-408, window :224-225): score =
// (q.k) * scale over keys [max(0, p - window + 1), p], softmax with the maximum
// subtracted, online over tiles of 32 keys so that no score matrix exists.
//
// One wave is one work item with 32 columns:
//   prompt   (heads that are no multiple of 32 or above 128, pages that are no multiple of 16 or very large, many short chains of tiles: see
//            f32_prompt_shared; the others run on attention_f32_prompt.hpp)
//            32 consecutive tokens of one request and one head: column c is
//            token t0 + c, each with its own causal bound
//   decode   one token, one KV head and up to 32 query heads of its group:
//            column c is head c, all with the token's bound; the token's keys
//            are cut into slices, a wave takes one and leaves a partial result
//            (maximum, sum, unnormalised output) that a second kernel merges (the
//            workgroup itself where its four waves hold all slices)
// A key tile is then read once for all 32 columns.
//
// MFMA 32x32x2 (lane l, g = l/32, c = l%32): A[c][g], B[g][c], D[8(i/4) + 4g +
// i%4][c] in accumulator register i.  Which element of the inner dimension a
// lane's operand stands for is free as long as A and B agree, so a lane reads
// four consecutive floats (16 bytes) and issues four MFMAs, one per float.
//   scores  S^T = K Q^T: A = key row c of the tile, floats 8kk + 4g .. + 3 of
//           head_dim, straight from the page; B = the same floats of column c's
//           query, from LDS.  The lane then holds, of column c, the scores of
//           keys 8(i/4) + 4g + i%4.
//   values  O^T += V^T P^T: A = values [head_dim row 32r + c][keys 8j + 4g .. +
//           3], one 16-byte read of the [head_dim][slot] value layout; B = the
//           probabilities of exactly those keys, which are registers 4j .. 4j +
//           3 of the scores.
//
// Loads carry no branch: a key outside the range the item reads is replaced by
// one inside it (a valid page) and masked (scores) or zeroed (values), so that
// pages given back behind a window or slots not yet written are never read.
// The next tile's keys are on their way during softmax and values, this tile's
// values during its scores (head sizes up to 128; larger ones load in turn,
// for registers).
#include <math.h>

#include "attention_f32.hpp"
#include "attention_f32_prompt.hpp"
#include "attention_merge.hpp"
#include "common.hpp"
#include "kllm_kernels.h"

namespace kllm {

constexpr int kF32Waves = 4;

struct AttnF32Args {
  const float* q;
  float* out;
  float* part;
  const float* cache;
  const int* positions;        // decode
  const int* span_of_token;    // decode
  const int* token_list;       // decode: the tokens (null: 0 .. count - 1)
  const int* query_tiles;      // prompt
  const int* span_start;       // prompt
  const int* span_pos;         // prompt
  const int* block_table;
  int count;                   // decode: tokens; prompt: blocks of 128
  int max_pages, page_size, H, KV, hd, window;
  int chunk;                   // a chunked mask (0: none)
  const float* sinks;          // per head: the score of one more key that has no value (null: none)
  OutGate gate;                // on the output (none: no sums)
  float scale;
  const float* slopes;         // per head: a bias that grows with the distance to the key (null: none)
  int nslices, col_blocks;     // decode: slices of the keys, blocks of 32 heads per group
  int wg_merge;                // decode: a workgroup's four slices leave one partial result
};

template <int HDT, bool DECODE>   // head_dim <= 32 * HDT
__global__ __launch_bounds__(64 * kF32Waves) void attn_f32_mfma_kernel(const AttnF32Args a) {
  constexpr int KC = 4 * HDT;                   // chunks of 8 floats of head_dim, at most
  constexpr bool AHEAD = HDT <= 4;              // next keys in flight while this tile is multiplied
  extern __shared__ __attribute__((aligned(16))) float q_lds[];   // [waves][32][hd + 4]
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 32, c = lane % 32;
  const int hd = a.hd, H = a.H, KV = a.KV, G = H / KV, page_size = a.page_size, window = a.window;
  const int kc = hd / 8;
  const int QLD = hd + 4;
  float* qs = q_lds + wave * 32 * QLD;
  const long item = (long)blockIdx.x * kF32Waves + wave;

  // ---- what this wave takes (the same in every lane)
  bool live;
  int t_base = 0, ncol = 1, h_base = 0, kvh = 0, span = 0, pos_base = 0, slice = 0;
  if (DECODE) {
    const long total = (long)a.count * KV * a.col_blocks * a.nslices;
    live = item < total;
    if (live) {
      slice = (int)(item % a.nslices);
      long r = item / a.nslices;
      const int cb = (int)(r % a.col_blocks);
      r /= a.col_blocks;
      kvh = (int)(r % KV);
      const int ti = (int)(r / KV);
      t_base = a.token_list ? a.token_list[ti] : ti;
      span = a.span_of_token[t_base];
      pos_base = a.positions[t_base];
      h_base = kvh * G + cb * 32;
      ncol = min(32, G - cb * 32);
    }
  } else {
    const long total = (long)a.count * 4 * H;
    live = item < total;
    if (live) {
      // Later tokens read more keys.  The later half of the (block, 32 tokens) pairs is
      // started first, longest first, then the earlier half, shortest first: a CU that
      // holds a workgroup of each half gets a long and a short one.
      const int h = (int)(item % H), place = (int)(item / H);
      const int npairs = a.count * 4, n_late = (npairs + 1) / 2;
      const int pair = place < n_late ? npairs - 1 - place : place - n_late;
      const int blk = pair / 4, sub = pair % 4;
      const int t0 = a.query_tiles[2 * blk] + 32 * sub;
      span = a.query_tiles[2 * blk + 1];
      const int s_begin = a.span_start[span], s_end = a.span_start[span + 1];
      if (t0 >= s_end) {
        live = false;                           // the block ends before these 32 tokens
      } else {
        t_base = t0;
        ncol = min(32, s_end - t0);
        pos_base = a.span_pos[span] + (t0 - s_begin);
        h_base = h;
        kvh = h / G;
      }
    }
  }

  // ---- the columns' queries into LDS
  if (live) {
    const int chunks = hd / 4;
    for (int idx = lane; idx < 32 * chunks; idx += kWave) {
      const int col = idx / chunks, ch = idx % chunks;
      const int cc = min(col, ncol - 1);
      const int tok = DECODE ? t_base : t_base + cc;
      const int head = DECODE ? h_base + cc : h_base;
      const floatx4 v = *reinterpret_cast<const floatx4*>(a.q + ((long)tok * H + head) * hd + 4 * ch);
      *reinterpret_cast<floatx4*>(qs + col * QLD + 4 * ch) = v;
    }
  }
  __syncthreads();
  if (!live) return;

  const bool col_ok = c < ncol;
  const int cc = min(c, ncol - 1);
  const int my_tok = DECODE ? t_base : t_base + cc;
  const int my_head = DECODE ? h_base + cc : h_base;
  const int my_pos = DECODE ? pos_base : pos_base + cc;
  const int my_start = first_key(my_pos, window, a.chunk);
  const float my_slope = a.slopes ? a.slopes[my_head] : 0.f;
  const int qmax = DECODE ? pos_base : pos_base + ncol - 1;            // last key any column reads
  const int lowest = first_key(pos_base, window, a.chunk);             // first key any column reads
  const int first = lowest / 32 * 32;
  const int tiles = (qmax - first) / 32 + 1;
  const int nslices = DECODE ? a.nslices : 1;
  const int per = (tiles + nslices - 1) / nslices;
  const int tile0 = slice * per, tile1 = min(tile0 + per, tiles);
  const int first_page_key = lowest / page_size * page_size;           // pages before this may be gone

  const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  auto page_index = [&](int key) { return page_shift >= 0 ? key >> page_shift : key / page_size; };
  auto page_slot = [&](int key) { return page_shift >= 0 ? key & (page_size - 1) : key % page_size; };
  auto inside = [&](int key) { return min(max(key, first_page_key), qmax); };   // a key whose page exists
  const int* table = a.block_table + (long)span * a.max_pages;
  const long block = (long)page_size * hd;
  const float* kcache = a.cache + (long)kvh * block;                   // + page * 2 * KV * block
  const float* vcache = a.cache + ((long)KV + kvh) * block;
  const long page_stride = 2L * KV * block;

  // A sink is where the running maximum and sum of the first slice start; one of a column's
  // two lanes holds its term, 1.
  const bool owns_sink = a.sinks && slice == 0;
  float m = owns_sink ? a.sinks[my_head] : -INFINITY, l = (owns_sink && g == 0) ? 1.f : 0.f;
  floatx16 acc[HDT];
#pragma unroll
  for (int r = 0; r < HDT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.f;

  struct VPages {
    int page[4];
  };
  auto lookup_k = [&](int tile) -> int { return table[page_index(inside(first + 32 * tile + c))]; };
  auto lookup_v = [&](int tile) -> VPages {
    VPages P;
#pragma unroll
    for (int j = 0; j < 4; ++j) P.page[j] = table[page_index(inside(first + 32 * tile + 8 * j + 4 * g) & ~3)];
    return P;
  };
  auto fetch_k = [&](int tile, int page, floatx4 (&K)[KC]) {
    const int key = inside(first + 32 * tile + c);
    const float* row = kcache + page * page_stride + (long)page_slot(key) * hd + 4 * g;
#pragma unroll
    for (int kk = 0; kk < KC; ++kk) K[kk] = *reinterpret_cast<const floatx4*>(row + 8 * min(kk, kc - 1));
  };
  auto fetch_v = [&](int tile, const VPages& P, floatx4 (&V)[HDT][4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key0 = inside(first + 32 * tile + 8 * j + 4 * g) & ~3;
      const float* base = vcache + P.page[j] * page_stride + page_slot(key0);
#pragma unroll
      for (int r = 0; r < HDT; ++r)
        V[r][j] = *reinterpret_cast<const floatx4*>(base + (long)min(32 * r + c, hd - 1) * page_size);
    }
  };

  floatx16 s;
  auto scores = [&](const floatx4 (&K)[KC]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KC; ++kk) {
      if (kk < kc) {
        const floatx4 b = *reinterpret_cast<const floatx4*>(qs + c * QLD + 8 * kk + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(K[kk][e], b[e], s, 0, 0, 0);
      }
    }
  };
  // mask, running maximum and sum; s becomes the probabilities
  auto softmax = [&](int tile) {
    const int kb = first + 32 * tile;
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kb + 8 * (i / 4) + 4 * g + i % 4;
      const bool ok = key <= my_pos && key >= my_start;
      float sc = s[i] * a.scale;
      if (a.slopes) sc -= my_slope * (float)(my_pos - key);   // (the same in every lane: a model without slopes skips it)
      s[i] = ok ? sc : -INFINITY;
      tmax = fmaxf(tmax, s[i]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
    const float m_new = fmaxf(m, tmax);
    const float mref = (m_new == -INFINITY) ? 0.f : m_new;   // a column with no key yet
    const float alpha = expf(m - mref);                      // exp(-inf) = 0
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = expf(s[i] - mref);
      psum += s[i];
    }
    l = l * alpha + psum;
    m = m_new;
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][i] *= alpha;
  };
  auto values = [&](int tile, floatx4 (&V)[HDT][4]) {
    const int kb = first + 32 * tile;
    if (kb < first_page_key || kb + 31 > qmax) {            // slots that were replaced or may hold anything
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = kb + 8 * j + 4 * g + e;
          const bool ok = key >= first_page_key && key <= qmax;
#pragma unroll
          for (int r = 0; r < HDT; ++r) V[r][j][e] = ok ? V[r][j][e] : 0.f;
        }
    }
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[r] = __builtin_amdgcn_mfma_f32_32x32x2f32(V[r][j][e], s[4 * j + e], acc[r], 0, 0, 0);
  };

  if (tile0 < tile1) {
    floatx4 K[KC];
    floatx4 V[HDT][4];
    if (AHEAD) {
      int kp = lookup_k(tile0);
      VPages vp = lookup_v(tile0);
      fetch_k(tile0, kp, K);
      kp = lookup_k(tile0 + 1);
      for (int tile = tile0; tile < tile1; ++tile) {
        fetch_v(tile, vp, V);
        vp = lookup_v(tile + 1);
        scores(K);
        fetch_k(tile + 1, kp, K);                            // a tile beyond the last: valid addresses, dropped
        kp = lookup_k(tile + 2);
        softmax(tile);
        values(tile, V);
      }
    } else {
      for (int tile = tile0; tile < tile1; ++tile) {
        fetch_k(tile, lookup_k(tile), K);
        const VPages vp = lookup_v(tile);
        scores(K);
        fetch_v(tile, vp, V);
        softmax(tile);
        values(tile, V);
      }
    }
  }
  l += __shfl_xor(l, 32, kWave);
  if (DECODE && a.wg_merge) {
    // The four waves of a workgroup hold four neighbouring slices of the same token and heads
    // (the number of slices is a multiple of four): they meet in LDS, each in the place of its
    // queries, and leave one partial result, so that the second kernel reads a quarter; four slices
    // in all are the result.
    if (col_ok) {
#pragma unroll
      for (int r = 0; r < HDT; ++r)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int d = 32 * r + 8 * b + 4 * g;
          if (d < hd) {
#pragma unroll
            for (int j = 0; j < 4; ++j) qs[c * QLD + d + j] = acc[r][4 * b + j];
          }
        }
      if (g == 0) {
        qs[c * QLD + hd] = m;                                // -inf and 0 for a slice without keys
        qs[c * QLD + hd + 1] = l;
      }
    }
    __syncthreads();
    const int nout = nslices / kF32Waves, sout = slice / kF32Waves;
    for (int idx = threadIdx.x; idx < ncol * hd; idx += 64 * kF32Waves) {
      const int col = idx / hd, d = idx % hd;
      float mw[kF32Waves], M = -INFINITY;
#pragma unroll
      for (int w = 0; w < kF32Waves; ++w) {
        mw[w] = q_lds[(w * 32 + col) * QLD + hd];
        M = fmaxf(M, mw[w]);
      }
      float o = 0.f, L = 0.f;
#pragma unroll
      for (int w = 0; w < kF32Waves; ++w) {
        const float wt = mw[w] == -INFINITY ? 0.f : expf(mw[w] - M);
        o += wt * q_lds[(w * 32 + col) * QLD + d];
        L += wt * q_lds[(w * 32 + col) * QLD + hd + 1];
      }
      if (nout == 1) {                                       // all of the token's keys: nothing is left to merge
        a.out[((long)t_base * H + h_base + col) * hd + d] = o / L * out_gate(a.gate, t_base, h_base + col, d);
        continue;
      }
      float* prow = a.part + (((long)t_base * H + h_base + col) * nout + sout) * (hd + 2);
      prow[d] = o;
      if (d == 0) {
        prow[hd] = M;
        prow[hd + 1] = L;
      }
    }
    return;
  }
  if (!col_ok) return;

  // acc[r][i] is output element 32r + 8(i/4) + 4g + i%4 of this lane's column
  if (nslices == 1) {
    const float inv = 1.f / l;                               // finite: a column reads its own key
    float* orow = a.out + ((long)my_tok * H + my_head) * hd;
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int d = 32 * r + 8 * b + 4 * g;
        if (d < hd) {
          const floatx4 og = out_gate4(a.gate, my_tok, my_head, d);
          floatx4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = acc[r][4 * b + j] * inv * og[j];
          *reinterpret_cast<floatx4*>(orow + d) = v;
        }
      }
    return;
  }
  float* prow = a.part + (((long)my_tok * H + my_head) * nslices + slice) * (hd + 2);
#pragma unroll
  for (int r = 0; r < HDT; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int d = 32 * r + 8 * b + 4 * g;
      if (d < hd) {
#pragma unroll
        for (int j = 0; j < 4; ++j) prow[d + j] = acc[r][4 * b + j];
      }
    }
  if (g == 0) {
    prow[hd] = m;                                            // -inf and 0 for a slice without keys
    prow[hd + 1] = l;
  }
}

// ---- Decode tokens with up to 16 query heads to a KV head, head sizes 32, 64, 96 and 128 and pages of a multiple of 16 slots:
// one wave takes one slice of the keys for the group's heads as 16 columns (MFMA 16x16x4: A[c][g], B[g][c], D[4g + i][c] for lane
// l, g = l / 16, c = l % 16), which is half the matrix instructions that 32 columns take.  Formulas and precision as above.
//   scores  A = key row c, floats 16kk + 4g ... + 3 of head_dim, one 16-byte read for four instructions; B = the same floats of
//           column c's query, in registers.  Row c of the u-th of two is key 8 (c / 4) + 4u + c % 4 of a tile of 32: the lane then holds
//           the scores of keys 8g ... 8g + 7.
//   values  A = values [head_dim row 16r + c][keys 8g ... 8g + 7], two 16-byte reads for eight instructions.
// What bounds it: up to a few tiles a wave, three trips to memory in a row (position and span; all pages of the wave's tiles, a half of a tile to a
// lane; keys and values) and the matrix instructions of its tiles; at many tokens the cache's bytes.  So the arguments come with the
// launch (the first eight), nothing goes through LDS before the merge, the sums are rescaled only where a maximum moved, and the slices are
// cut over the waves of the workgroups that a launch has, without 64-bit divisions.  us in a step, 32 columns before and 16 now: 8 tokens
// at 1,400 keys, 4 KV heads of 64 16.0 -> 9.1, of which the multiplications of two tiles are 1.7 (on 32 columns 3.4); steps of 1.1B Llama sizes, 1 / 8 / 16 / 32 tokens
// 1,394 / 1,502 / 1,701 / 2,860 -> 1,271 / 1,350 / 1,551 / 2,663, of 7B (2 tokens) 5,910 -> 5,665, of 8B (4) 6,470 -> 6,220.
// (Those with exponentials as exp2 of one rounded product with log2(e), whose error grows with a score's distance to the maximum: 2^-24 of it, 60 units of a
// weight's last place for scores 80 apart.  expf is within 1.4 units of 2^-24; it costs 0.6 us of 10.2 at 8 tokens and
// 1,400 keys, 0.9 of 24.1 at 64 tokens and 1,000, and of the steps of 1 / 8 / 16 / 32 tokens 0.6 / 0.5 / 0.7 / 0.5 %.  exp_negative, within 2.3: 11.1 -> 10.8 and 22.7 -> 22.4,
// 16 heads of 32, 16 tokens at 4,000 39.6 -> 42.2; no step of 1.1B sizes shows it.)
template <int HDT>   // head_dim = 16 * HDT
__global__ __launch_bounds__(64 * kF32Waves) __attribute__((amdgpu_waves_per_eu(HDT <= 4 ? 2 : 1))) void attn_f32_decode_kernel(
    const float* __restrict__ cache, const int* __restrict__ positions, const int* __restrict__ span_of_token, const int* __restrict__ block_table,
    const int* __restrict__ token_list, const float* __restrict__ q, int max_pages, int KV, float* __restrict__ out, float* __restrict__ part, int H, int G,
    int page16, int wgs, unsigned page_magic, unsigned slice_magic, int window, int chunk, const float* __restrict__ sinks, float scale,
    const float* __restrict__ slopes, const OutGate gate) {
  constexpr int hd = 16 * HDT;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 16, c = lane % 16;
  int at = blockIdx.x;                                       // (vector loads: scalar ones come one behind the other)
  asm volatile("" : "+v"(at));
  if (token_list) at = token_list[at];
  const int pos_v = positions[at], span_v = span_of_token[at];
  asm volatile("" ::"s"(H), "s"(G), "s"(page16), "s"(wgs), "s"(page_magic), "s"(slice_magic), "s"(window), "s"(chunk), "s"(sinks), "s"(scale),
               "s"(slopes), "s"(out), "s"(part), "s"(gate.sums));
  const int t = __builtin_amdgcn_readfirstlane(at), page_size = 16 * page16, kvh = blockIdx.y;
  const int nslices = wgs * kF32Waves, slice = blockIdx.z * kF32Waves + wave;
  const bool head_ok = c < G;
  const int head = kvh * G + (head_ok ? c : 0);              // (a column without a head computes another's, and nothing comes of it)
  const float slope = slopes ? slopes[head] : 0.f;
  floatx4 qb[HDT];
#pragma unroll
  for (int kk = 0; kk < HDT; ++kk) qb[kk] = *reinterpret_cast<const floatx4*>(q + ((long)t * H + head) * hd + 16 * kk + 4 * g);

  const int len = __builtin_amdgcn_readfirstlane(pos_v) + 1, span = __builtin_amdgcn_readfirstlane(span_v);
  const int start = first_key(len - 1, window, chunk), first = start & ~31;
  const int tiles = (len - first + 31) / 32;
  unsigned left;
  const int per = (int)divided((unsigned)(tiles + nslices - 1), (unsigned)nslices, slice_magic, left);
  const int tile0 = slice * per, tile1 = min(tile0 + per, tiles);
  const int* table = block_table + (long)span * max_pages;
  const long block = (long)page_size * hd;

  // A sink is where the running maximum and sum of the first slice start; one of a column's four lanes holds its term, 1.
  const bool owns_sink = sinks && slice == 0;
  float m = owns_sink ? sinks[head] : -INFINITY, l = (owns_sink && g == 0) ? 1.f : 0.f;
  floatx4 acc[HDT];
#pragma unroll
  for (int r = 0; r < HDT; ++r) acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};

  struct Tile {
    floatx4 k[2][HDT], v[HDT][2];
    unsigned mask;             // which of its keys are read (0: there is no such tile)
  };
  auto bits = [](int lo, int hi) -> unsigned {               // lo ... hi - 1 of 32 (lo < hi)
    return (~0u >> (32 - min(max(hi, 1), 32))) & (~0u << min(max(lo, 0), 31));
  };
  // Where the 64 halves (16 keys, of one page) of 32 tiles from b0 on lie, a half to a lane.  One that is not read (its page may be
  // gone) reads page 0, whose keys and values nothing comes of.
  struct Places {
    unsigned mask;
    int slot;
    long base;               // floats from the cache's first to the page's keys of this head
  };
  auto lookup = [&](int b0) -> Places {
    Places P;
    const int tile = b0 + lane / 2, kb = first + tile * 32;
    P.mask = tile < tile1 ? bits(start - kb, len - kb) : 0u;
    const bool live = (P.mask >> (16 * (lane % 2))) & 0xFFFFu;
    unsigned left;
    const int index = (int)divided(live ? (unsigned)kb / 16 + lane % 2 : 0u, (unsigned)page16, page_magic, left);
    const int page = table[index];
    P.slot = (int)left * 16;
    P.base = ((long)(live ? page : 0) * 2 * KV + kvh) * block;
    return P;
  };
  const int k_lane = (8 * (c / 4 % 2) + c % 4) * hd + 4 * g;             // floats of this lane in a half's keys
  const int v_lane = c * page_size + 8 * (g % 2);                        // ... and in a page's values
  auto fetch = [&](const Places& P, int i) -> Tile {         // the i-th of those tiles
    Tile T;
    T.mask = __builtin_amdgcn_readlane(P.mask, 2 * i);
    const float* kp[2];
    const float* vp[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned lo = __builtin_amdgcn_readlane((int)P.base, 2 * i + h);
      const long base = (long)((unsigned long)(unsigned)__builtin_amdgcn_readlane((int)(P.base >> 32), 2 * i + h) << 32 | lo);
      const int slot = __builtin_amdgcn_readlane(P.slot, 2 * i + h);
      kp[h] = cache + base + slot * hd;
      vp[h] = cache + base + KV * block + slot;
    }
    __builtin_amdgcn_sched_barrier(0);
    const float* kl = (c < 8 ? kp[0] : kp[1]) + k_lane;
    const float* vl = (g < 2 ? vp[0] : vp[1]) + v_lane;
#pragma unroll
    for (int kk = 0; kk < HDT; ++kk)
#pragma unroll
      for (int u = 0; u < 2; ++u) T.k[u][kk] = *reinterpret_cast<const floatx4*>(kl + 4 * u * hd + 16 * kk);
    __builtin_amdgcn_sched_barrier(0);     // (keys first: the scores wait for no values)
#pragma unroll
    for (int r = 0; r < HDT; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) T.v[r][h] = *reinterpret_cast<const floatx4*>(vl + (long)r * 16 * page_size + 4 * h);
    __builtin_amdgcn_sched_barrier(0);
    return T;
  };
  auto compute = [&](Tile& T, int tile) {
    floatx4 s[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < HDT; ++kk)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < 2; ++u) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(T.k[u][kk][e], qb[kk][e], s[u], 0, 0, 0);
    float sc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sc[e] = s[e / 4][e % 4] * scale;
    if (slopes) {
      const int far = len - 1 - (first + tile * 32) - 8 * g;
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] -= slope * (float)(far - e);
    }
    if (T.mask != ~0u) {                                     // first and last tiles: what is not read may hold anything
      const unsigned mine = T.mask >> (8 * g);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool ok = (mine >> e) & 1u;
        sc[e] = ok ? sc[e] : -INFINITY;
#pragma unroll
        for (int r = 0; r < HDT; ++r) T.v[r][e / 4][e % 4] = ok ? T.v[r][e / 4][e % 4] : 0.f;
      }
    }
    float tmax = sc[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) tmax = fmaxf(tmax, sc[e]);
    const float m_new = fmaxf(m, group4_max(tmax));
    const float mref = m_new == -INFINITY ? 0.f : m_new;     // scores may have overflowed
    const float alpha = expf(m - mref);                      // exp(-inf) = 0
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sc[e] = expf(sc[e] - mref);
      psum += sc[e];
    }
    l = l * alpha + psum;
    if (__builtin_amdgcn_ballot_w64(m_new > m)) {            // (after a few tiles the maximum rarely moves)
#pragma unroll
      for (int r = 0; r < HDT; ++r) acc[r] *= alpha;
    }
    m = m_new;
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int r = 0; r < HDT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(T.v[r][e / 4][e % 4], sc[e], acc[r], 0, 0, 0);
  };
  // While a tile is multiplied the next one's operands are on their way, in two buffers by name.  Beyond the wave's last tile that
  // one is asked for again.
  for (int b0 = tile0; b0 < tile1; b0 += 32) {
    const Places P = lookup(b0);
    const int n = min(tile1 - b0, 32);
    Tile A = fetch(P, 0), B;
    if (n == 1) {            // (short contexts: nothing is asked for that is not read)
      compute(A, b0);
      break;
    }
#pragma unroll 1
    for (int i = 0; i < n; i += 2) {
      B = fetch(P, min(i + 1, n - 1));
      compute(A, b0 + i);
      A = fetch(P, min(i + 2, n - 1));
      if (i + 1 < n) compute(B, b0 + i + 1);
    }
  }
  l = group4_sum(l);

  // ---- the waves' results meet in LDS; a thread merges, in the order of the waves, four elements of one head: the output itself
  // where this workgroup had all the keys, else the workgroup's partial result
  extern __shared__ __attribute__((aligned(16))) float red[];   // [waves][G][hd + 4]
  constexpr int RS = hd + 4;
  if (head_ok) {
    float* mine = red + (wave * G + c) * RS;
#pragma unroll
    for (int r = 0; r < HDT; ++r) *reinterpret_cast<floatx4*>(mine + 16 * r + 4 * g) = acc[r];
    if (g == 0) {
      mine[hd] = m;                                          // -inf and 0 for a slice without keys
      mine[hd + 1] = l;
    }
  }
  __syncthreads();
  constexpr int CH = hd / 4;
  for (int idx = threadIdx.x; idx < G * CH; idx += 64 * kF32Waves) {
    const int hc = idx / CH, d4 = (idx % CH) * 4;
    const float* col = red + hc * RS;
    float mj[kF32Waves], M = -INFINITY;
#pragma unroll
    for (int j = 0; j < kF32Waves; ++j) {
      mj[j] = col[j * G * RS + hd];
      M = fmaxf(M, mj[j]);
    }
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
#pragma unroll
    for (int j = 0; j < kF32Waves; ++j) {
      const float* w = col + j * G * RS;
      const float wj = M != -INFINITY ? expf(mj[j] - M) : 0.f;
      L += wj * w[hd + 1];
      v += wj * *reinterpret_cast<const floatx4*>(w + d4);
    }
    const long row = (long)t * H + kvh * G + hc;
    if (wgs == 1) {
      const floatx4 og = out_gate4(gate, t, kvh * G + hc, d4);
      const float inv = 1.f / L;                             // finite: a column reads its own key
      floatx4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = v[j] * inv * og[j];
      *reinterpret_cast<floatx4*>(out + row * hd + d4) = o;
    } else {
      float* prow = part + (row * wgs + blockIdx.z) * (hd + 2);   // 8-byte rows
      *reinterpret_cast<floatx2*>(prow + d4) = floatx2{v[0], v[1]};
      *reinterpret_cast<floatx2*>(prow + d4 + 2) = floatx2{v[2], v[3]};
      if (d4 == 0) *reinterpret_cast<floatx2*>(prow + hd) = floatx2{M, L};
    }
  }
}

template <int HDT>
static void launch_f32_decode(const AttnF32Args& a, int wgs, hipStream_t stream) {
  const int G = a.H / a.KV;
  const unsigned page16 = a.page_size / 16, slices = wgs * kF32Waves;
  const unsigned page_magic = page16 == 1 ? 0xFFFFFFFFu : (unsigned)((1ull << 32) / page16), slice_magic = (unsigned)((1ull << 32) / slices);
  hipLaunchKernelGGL(attn_f32_decode_kernel<HDT>, dim3(a.count, a.KV, wgs), dim3(64 * kF32Waves),
                     (size_t)kF32Waves * G * (16 * HDT + 4) * sizeof(float), stream, a.cache, a.positions, a.span_of_token, a.block_table, a.token_list,
                     a.q, a.max_pages, a.KV, a.out, a.part, a.H, G, (int)page16, wgs, page_magic, slice_magic, a.window, a.chunk, a.sinks, a.scale,
                     a.slopes, a.gate);
}

template <int HDT, bool DECODE>
static int launch_f32(const AttnF32Args& a, long items, hipStream_t stream) {
  const size_t lds = (size_t)kF32Waves * 32 * (a.hd + 4) * sizeof(float);
  static int raised = 0;
  if (lds > 64 * 1024 && !raised) {
    hipError_t e = hipFuncSetAttribute((const void*)attn_f32_mfma_kernel<HDT, DECODE>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) KLLM_FAIL((int)e, "attention float32: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = 1;
  }
  const long grid = (items + kF32Waves - 1) / kF32Waves;
  KLLM_REQUIRE(grid > 0 && grid < (1L << 31), "attention float32: %ld work items do not fit a grid", items);
  hipLaunchKernelGGL((attn_f32_mfma_kernel<HDT, DECODE>), dim3((unsigned)grid), dim3(64 * kF32Waves), lds, stream, a);
  return 0;
}

template <bool DECODE>
static int dispatch_f32(const AttnF32Args& a, long items, hipStream_t stream) {
  const int hdt = (a.hd + 31) / 32;
  if (hdt <= 1) return launch_f32<1, DECODE>(a, items, stream);
  if (hdt <= 2) return launch_f32<2, DECODE>(a, items, stream);
  if (hdt <= 3) return launch_f32<3, DECODE>(a, items, stream);
  if (hdt <= 4) return launch_f32<4, DECODE>(a, items, stream);
  if (hdt <= 6) return launch_f32<6, DECODE>(a, items, stream);
  return launch_f32<8, DECODE>(a, items, stream);
}

bool attn_f32_fits(int hd, int page_size) {
  return hd >= 8 && hd <= 256 && hd % 8 == 0 && page_size > 0 && page_size % 4 == 0;
}

extern "C" int kllm_attn_f32_fits(int hd, int page_size) { return attn_f32_fits(hd, page_size) ? 1 : 0; }

// Whether a decode token's keys go by attn_f32_decode_kernel, on 16 columns.
static bool f32_sixteen(int H, int KV, int hd, int page_size) {
  return H / KV <= 16 && hd % 32 == 0 && hd <= 128 && page_size % 16 == 0 && KV <= 65535;
}

int attn_f32_slices(int n, int KV, int H, int hd, int max_keys, int page_size) {
  // About four waves per CU across the chip, shared out over tokens x KV heads x blocks of 32 heads; a slice is one wave and should have
  // 32 keys at least (one token at 32,768 keys 47 us with 256 against 69 with 64, on 32 columns; on 16, in us with the merge in a replayed graph:
  // 8 tokens x 4 KV heads of 64 at 1,000 keys 17.1 / 13.0 / 10.0 / 7.5 / 7.9 with 4 / 8 / 16 / 32 / 64; 16 x 8 of 128 41.6 / 30.9 / 37.3 / 35.2 / 40.1).
  const int col_blocks = (H / KV + 31) / 32;
  const long groups = (long)n * KV * col_blocks;
  const int cus = device_cus();
  long want = (groups >= cus ? 8L : 4L) * cus / (groups > 0 ? groups : 1);
  const long keys = max_keys > 0 ? max_keys : 2048;          // (of a table's width, up to twice the context's)
  if (groups >= cus && f32_sixteen(H, KV, hd, page_size)) {
    // From one group per CU on, on 16 columns, the four slices of one workgroup, which leave nothing to merge (4 / 8 slices: 64 tokens x 4 KV heads of 64 at 250
    // keys 9.8 / 10.9, at 32,768 742 / 746; 8 x 32 of 128 at 250 19.9 / 20.7, at 6,000 282 / 286).  Unless the CUs' last round of workgroups is at least
    // half empty and the keys are many: then eight, or sixteen, where that shortens it once more (4 / 8 / 16 slices, groups per CU 1 1/8, 1 1/2, 2 1/8, 3 1/2: heads of 64
    // at 2,048 keys 70.7 / 60.6 / 56.0, 80.2 / 75.4 / 77.2, 120 / 110 / 107, 171 / 167 / 170, at 6,000 222 / 183 / 169, 238 / 211 / 212, 354 / 322 / 297,
    // 501 / 481 / 464; of 128 at 2,048 169 / 143 / 139, 175 / 157 / 172, 265 / 246 / 254, 375 / 352 / 385, at 6,000 479 / 386 / 338, 499 / 424 / 420, 747 /
    // 659 / 632, 1,035 / 967 / 989; 4 / 8 at 600 59.8 / 57.1, 61.6 / 64.1, 95.1 / 99.9, 136 / 152, at 1,000 85.8 / 79.2, 95.1 / 90.6, 143 / 141, 197 / 205).
    auto rounds = [&](long workgroups) { return ceil_div(groups * workgroups, cus); };
    const bool few = 4 * groups <= 5L * cus;                 // a quarter of a second round at most
    want = kF32Waves;
    if (groups <= 4L * cus && keys >= (few ? 1024 : 2048) && rounds(2) < 2 * rounds(1))
      want = (keys >= (few ? 4096 : 8192) && rounds(4) < 2 * rounds(2) ? 4 : 2) * kF32Waves;
  } else if (groups == cus && H / KV <= 16 && hd % 32 == 0 && hd <= 128 && (hd > 64 || keys <= 768)) {
    // On 32 columns eight waves a CU (heads of 64, pages of 20 slots, 4 / 8 slices: at 1,000 keys 41.2 / 40.7, at 6,000 200 / 182; of 128, 1 1/8 groups per
    // CU, 4 / 7: at 2,048 222 / 158), but in whole rounds four of large heads (128, one group per CU: at 600 46.0 / 63.4, at 6,000 321 / 335) and of few
    // keys (64: at 250 16.4 / 19.2, at 600 28.2 / 31.9).
    want = kF32Waves;
  }
  long most = max_keys > 0 ? max_keys / 32 : 64;
  if (most > kAttnF32MaxSlices) most = kAttnF32MaxSlices;
  // Up to 128 keys (a tile of 32 a wave) the second kernel costs more than the keys: one workgroup's four
  // slices, which write the output (8 tokens x 4 KV heads of 64, in us, in a replayed graph: 64 keys 10.0, with two
  // slices and the merge 11.5; 128 keys 10.4 against 12.5; 8 KV heads of 128: 14.4 against 17.0, 16.1 against
  // 18.5).  Beyond it the matrix products of a second tile on the same SIMDs cost what the merge does (256 keys: 13.4
  // with four slices, 13.1 with eight waves to a workgroup, 12.2 with eight slices and the merge).  Up to 64 keys, where two of
  // the four waves have no tile, only while the workgroup's own merge is short (16 heads of 128 to a KV head, one token: 16.6
  // against 15.2; 32 of 64: 12.7 against 11.5; 4 of 128: 14.2 against 17.0) and the groups are no more than CUs (512: 27.3
  // against 18.6).  One tile of keys: one wave writes the output (8 tokens, 32 heads of 64 to a KV head: 9.9, in four slices 12.7).
  const int heads = H / KV < 32 ? H / KV : 32;
  const bool whole = max_keys > 64 ? max_keys <= 32 * kF32Waves : max_keys > 32 && heads * hd < 2048 && groups <= cus;
  if (whole && want >= kF32Waves) return kF32Waves;
  if (want > most) want = most;
  if (want < 1) want = 1;
  return (int)want;
}

int attn_f32_decode(const float* q, float* out, float* part, const float* cache, const int* positions,
                    const int* span_of_token, const int* block_table, int max_pages, int page_size,
                    int H, int KV, int hd, int window, int chunk, const float* sinks, float scale, const float* slopes, int nslices,
                    const int* token_list, int count, const OutGate& gate, hipStream_t stream) {
  KLLM_REQUIRE(attn_f32_fits(hd, page_size),
               "attn_decode float32: head_dim %d must be a multiple of 8 up to 256 and page_size %d a multiple of 4",
               hd, page_size);
  KLLM_REQUIRE(nslices >= 1 && nslices <= kAttnF32MaxSlices, "attn_decode float32: nslices %d is outside [1, %d]",
               nslices, kAttnF32MaxSlices);
  AttnF32Args a = {};
  a.q = q; a.out = out; a.part = part; a.cache = cache;
  a.positions = positions; a.span_of_token = span_of_token; a.token_list = token_list;
  a.block_table = block_table; a.count = count;
  a.max_pages = max_pages; a.page_size = page_size; a.H = H; a.KV = KV; a.hd = hd; a.window = window; a.chunk = chunk; a.sinks = sinks; a.gate = gate;
  a.scale = scale; a.slopes = slopes; a.nslices = nslices; a.col_blocks = (H / KV + 31) / 32;
  // The kernel of 16 columns takes a workgroup's four slices at a time, whatever their number (no more partial results than
  // the slices that ``part`` has room for).
  const int wgs = (nslices + kF32Waves - 1) / kF32Waves;
  if (f32_sixteen(H, KV, hd, page_size)) {
    if (hd == 32) launch_f32_decode<2>(a, wgs, stream);
    else if (hd == 64) launch_f32_decode<4>(a, wgs, stream);
    else if (hd == 96) launch_f32_decode<6>(a, wgs, stream);
    else launch_f32_decode<8>(a, wgs, stream);
    KLLM_CHECK_LAUNCH("attn_decode float32");
    if (wgs > 1) {
      launch_attn_merge<float>(out, part, count, H, hd, wgs, token_list, gate, stream);
      KLLM_CHECK_LAUNCH("attn_merge float32");
    }
    return 0;
  }
  a.wg_merge = nslices % kF32Waves == 0;
  const long items = (long)count * KV * a.col_blocks * nslices;
  if (int rc = dispatch_f32<true>(a, items, stream)) return rc;
  KLLM_CHECK_LAUNCH("attn_decode float32");
  if (nslices > 1 && nslices != kF32Waves) {
    launch_attn_merge<float>(out, part, count, H, hd, a.wg_merge ? nslices / kF32Waves : nslices, token_list, gate, stream);
    KLLM_CHECK_LAUNCH("attn_merge float32");
  }
  return 0;
}

template <int HDT>
static int launch_f32_prompt(const AttnF32Args& a, hipStream_t stream) {
  const size_t lds = (size_t)kF32Waves * 2 * F32PromptShape<HDT>::TB;
  static int raised = 0;
  if (lds > 64 * 1024 && !raised) {
    hipError_t e = hipFuncSetAttribute((const void*)attn_f32_prompt_kernel<HDT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) KLLM_FAIL((int)e, "attention float32: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = 1;
  }
  const long grid = (long)a.count * 4 * a.H;
  KLLM_REQUIRE(grid < (1L << 31), "attention float32: %ld work items do not fit a grid", grid);
  hipLaunchKernelGGL(attn_f32_prompt_kernel<HDT>, dim3((unsigned)grid), dim3(64 * kF32Waves), lds, stream, a.q, a.out, a.cache, a.query_tiles,
                     a.count, a.span_start, a.span_pos, a.block_table, a.max_pages, a.page_size, a.H, a.KV, a.window, a.chunk, a.sinks, a.scale,
                     a.slopes, a.gate);
  return 0;
}

// Which kernel takes a prompt: four waves to 32 tokens and a head (attn_f32_prompt_kernel), or one, four heads to a workgroup.  The former's chains of
// tiles are a quarter as long, but it has two workgroups a CU (heads of 64; one of 96 and 128), each with what it costs beside its tiles, also
// where the block of 128 ends before its 32 tokens.  So with more than two such parts a CU it needs chains: of some tiles, more with more parts and
// larger heads (us, one wave / four: 16 prompts of 40 tokens, 32 heads of 64 14.2 / 19.6, of 96 21.1 / 32.5; 29 of 6, 40 heads of 96 19 / 57; 64 of 64
// 22.6 / 33.6; 24 prompts of 51, 40 heads of 128 64 / 86; but 32 heads of 64, four of 500 72 / 68).  And for heads of 96 and 128 with four parts
// a CU and more, all of them alike, of more than three rounds of tiles (behind a window of 256, 2,048 tokens of 32 heads of 96 94 / 122, of 128 129 / 151, of 64
// heads 252 / 294; eight of 100 behind 300, 64 of 128 140 / 160; without a window 863 / 710).  Of 888 drawn sizes 69 were more than 3 %
// slower, up to three times, with the latter everywhere, 6 by this rule, up to 1.22; in the mean it gives 1.95, everywhere 1.94.  Without numbers of keys: four waves.
static bool f32_prompt_shared(int n_tiles, int H, int hd, int n_rows, long keys_total, int keys_longest, int window) {
  if (keys_total <= 0 || keys_longest <= 0) return true;
  const float cus = device_cus();
  const long parts = n_rows > 0 && n_rows / 32 + n_tiles < 4L * n_tiles ? n_rows / 32 + n_tiles : 4L * n_tiles;      // that have tokens
  float mean = (float)keys_total / n_tiles, most = keys_longest;
  if (window > 0) {                     // (the blocks' numbers are of 128 tokens)
    mean = fminf(mean, window + 48.f);
    most = fminf(most, window + 48.f);
  }
  mean = fmaxf((mean - 16.f * ((float)parts / n_tiles - 1.f)) / 32.f + 0.5f, 1.f);
  most = most / 32.f + 0.5f;
  const float all = 4.f * n_tiles * H / cus;
  if (all <= 2.f) return true;
  if (0.5f * (mean + most) < (hd > 32 ? 1.5f / 64 * hd : 0.f) + 0.5f * log2f(all)) return false;       // (heads of 32: four workgroups a CU)
  return !(hd >= 96 && parts * H >= 4 * cus && most <= 13.5f && mean >= 0.72f * most);
}

extern "C" int kllm_attn_f32_prompt_shared(int n_tiles, int H, int hd, int n_rows, long keys_total, int keys_longest, int window) {
  return n_tiles > 0 && f32_prompt_shared(n_tiles, H, hd, n_rows, keys_total, keys_longest, window) ? 1 : 0;
}

int attn_f32_prefill(const float* q, float* out, const float* cache, const int* query_tiles, int n_tiles,
                     const int* span_start, const int* span_pos, const int* block_table, int max_pages,
                     int page_size, int H, int KV, int hd, int window, int chunk, const float* sinks, float scale, const float* slopes,
                     long keys_total, int keys_longest, int n_rows, const OutGate& gate, hipStream_t stream) {
  KLLM_REQUIRE(attn_f32_fits(hd, page_size),
               "attn_prefill float32: head_dim %d must be a multiple of 8 up to 256 and page_size %d a multiple of 4",
               hd, page_size);
  AttnF32Args a = {};
  a.q = q; a.out = out; a.cache = cache;
  a.query_tiles = query_tiles; a.span_start = span_start; a.span_pos = span_pos;
  a.block_table = block_table; a.count = n_tiles;
  a.max_pages = max_pages; a.page_size = page_size; a.H = H; a.KV = KV; a.hd = hd; a.window = window; a.chunk = chunk; a.sinks = sinks; a.gate = gate;
  a.scale = scale; a.slopes = slopes; a.nslices = 1; a.col_blocks = 1;
  if (page_size % 16 == 0 && hd % 32 == 0 && hd <= 128 && direct_pages(cache, KV, hd, page_size, sizeof(float)) &&
      f32_prompt_shared(n_tiles, H, hd, n_rows, keys_total, keys_longest, window)) {
    const int rc = hd == 32 ? launch_f32_prompt<1>(a, stream) : hd == 64 ? launch_f32_prompt<2>(a, stream)
                 : hd == 96 ? launch_f32_prompt<3>(a, stream) : launch_f32_prompt<4>(a, stream);
    if (rc) return rc;
    KLLM_CHECK_LAUNCH("attn_prefill float32");
    return 0;
  }
  const long items = (long)n_tiles * 4 * H;
  if (int rc = dispatch_f32<false>(a, items, stream)) return rc;
  KLLM_CHECK_LAUNCH("attn_prefill float32");
  return 0;
}

}  // namespace kllm
