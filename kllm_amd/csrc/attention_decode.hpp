// Decode attention over the paged cache on the matrix cores (bfloat16).
//
// One wave takes one token, one KV head with up to 16 of its query heads, and
// one slice of the token's keys; it streams that slice's pages from memory
// once, for all heads of the group.  The waves of a workgroup (four or eight)
// merge their results in LDS.  Where one workgroup covers all keys of its token it writes the
// output itself; otherwise it leaves one partial result (running maximum, sum,
// unnormalised output) and a second kernel merges the workgroups' partials.
// The launch does not depend on any context length, so a recorded step can be
// replayed as contexts grow.
//
// Formulas as in the generic kernel (reference: backend/model.cu:343-408):
// score = (q.k)/sqrt(hd) over keys [max(0, p-window+1), p], softmax with the
// maximum subtracted, all in 32-bit; probabilities are rounded to bfloat16 for
// the product with the values and their sum is taken over the rounded numbers.
//
// MFMA 16x16x32 (lane l: g = l/16, c = l%16): A[c][8g..8g+7], B[8g..8g+7][c],
// D[4g+i][c].  Scores: A = 16 of a tile's 32 keys x 32 of hd (one key row per lane, straight
// from its page), B = q of 16 heads, D[key row 4g+i][head c].  Values: A = values [hd row c][8 keys], in the
// order in which a lane holds its probabilities.  Which key stands in which row of A is free: with key 8 (c / 4) + 4 u + c % 4 in
// row c of the u-th of two instructions a lane's probabilities are those of eight neighbouring keys, whose values are one
// 16-byte read from the [hd][slot] layout (two of 8 bytes before).
//
// What bounds it: at small batches three trips to memory in a row (position and span; pages; keys and values), then a
// tile's instructions, of which a wave alone on its SIMD issues one in four cycles or more; at large ones the cache's bytes.  So all pages of
// a wave's tiles are one load, a half of a tile to a lane, and come back lane by lane as scalars; masks are words that whole tiles skip;
// exponentials are the hardware's (base 2); the sums are rescaled only where a maximum moved; a wave without
// keys asks for none.  us in a step, the tile-by-tile lookups before and now: 8 tokens at 1,400 keys, 4 KV heads of 64 8.3 -> 5.5, one token at 540 6.2 ->
// 5.0, 64 tokens at 1,400 22 -> 18 (92 MB: 5.1 TB/s), 16 tokens with 8 KV heads of 128 23.5 -> 22.2.  A step of 1 / 8 / 64 tokens 793 / 866 / 1,480 -> 769 / 831 /
// 1,395 us, at 8B sizes of 16 tokens 3,860 -> 3,815, Natenex of 8 tokens 730 -> 704.
#pragma once

#include "attention_merge.hpp"
#include "common.hpp"

namespace kllm {

// KEPT: kept first positions behind the window (an instance of its own: the others carry none of it)
// TILED: the output's rows in the next product's order (gate.side; one instance for both cost the plain one 2 us of 49, in scalar registers)
// G: query heads of a KV head; page16: page size / 16; page_magic and slice_magic: see divided(), of page16 and of the slices (waves).
// The workgroup's place: the token (or its place in token_list), KV head and tile of its heads, and which of wgs workgroups.
template <int HDT, int kDecodeWaves, bool BIASED, bool KEPT, bool TILED>  // head_dim = 16 * HDT; BIASED: scores lose slope * distance
__device__ __forceinline__ void attn_decode_block(
    const bf16_t* __restrict__ cache, const int* __restrict__ positions, const int* __restrict__ span_of_token,
    const int* __restrict__ block_table, const int* __restrict__ token_list, const bf16_t* __restrict__ q, int max_pages, int KV,
    bf16_t* __restrict__ final_out, float* __restrict__ part, int H, int G, int page16, int wgs, unsigned page_magic, unsigned slice_magic, int window, int chunk,
    const float* __restrict__ sinks, int keep_first, float scale, const float* __restrict__ slopes, int head_tiles, const OutGate gate, int place_token, int place_head, int place_wg) {
  constexpr int hd = 16 * HDT;
  constexpr int KS = (hd + 31) / 32;           // MFMA steps over head_dim for the scores
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 16, c = lane % 16;
  // Trips to memory in a row are what a short launch is made of: the position and the span go out together at once (the first eight
  // arguments lie in registers when a wave starts), and the next trip is all pages of the wave's tiles.  (Vector loads, although
  // the address is the same in every lane: scalar ones come one behind the other as the compiler's registers fall.)
  int at = place_token;
  asm volatile("" : "+v"(at));
  if (token_list) at = token_list[at];
  const int pos_v = positions[at], span_v = span_of_token[at];
  asm volatile("" ::"s"(H), "s"(G), "s"(page16), "s"(page_magic), "s"(slice_magic), "s"(window), "s"(chunk), "s"(keep_first), "s"(scale),
               "s"(head_tiles), "s"(wgs), "s"(sinks), "s"(final_out), "s"(part), "s"(gate.sums), "s"(gate.side));
  const int t = __builtin_amdgcn_readfirstlane(at), page_size = 16 * page16;
  int kvh = place_head, ht = 0;
  if (head_tiles > 1) {
    kvh = place_head / head_tiles;
    ht = place_head % head_tiles;
  }
  const int nslices = wgs * kDecodeWaves;
  const int slice = place_wg * kDecodeWaves + wave;

  const int head_in_group = ht * 16 + c;                   // this lane's column
  const bool head_ok = head_in_group < G;
  const int head = kvh * G + (head_ok ? head_in_group : 0);
  const float slope = (BIASED && head_ok) ? slopes[head] * kLog2E : 0.f;   // a bias that grows with the distance to the key
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qb[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = 32 * ks + 8 * g;
    const bool there = hd % 32 == 0 || d0 < hd;            // (a column without a head computes another's, and nothing comes of it)
    qb[ks] = *reinterpret_cast<const bf16x8*>(q + ((long)t * H + head) * hd + (there ? d0 : 0));
    if (!there) qb[ks] = zero8;
  }

  const int len = __builtin_amdgcn_readfirstlane(pos_v) + 1, span = __builtin_amdgcn_readfirstlane(span_v);
  const int start = first_key(len - 1, window, chunk);     // window and chunked mask
  const int first = start & ~31;                           // tiles of 32 keys from here
  // Kept first positions: the keys below kept_end (none of them in the window's tiles) come
  // first, in n_kept tiles of their own from key 0; pages between them and the window may be gone.
  const int kept_end = KEPT ? min(keep_first, first) : 0;
  const int n_kept = KEPT ? (kept_end + 31) / 32 : 0;
  const int tiles = (len - first + 31) / 32 + n_kept;
  unsigned left;
  const int per = (int)divided((unsigned)(tiles + nslices - 1), (unsigned)nslices, slice_magic, left);
  const int tile0 = slice * per, tile1 = min(tile0 + per, tiles);
  const int* table = block_table + (long)span * max_pages;
  const long block = (long)page_size * hd;

  // Scores are in units of log2(e): a probability is one exponential of the hardware's.
  // A sink (a key with a score of its own and no value) is where the running maximum and
  // sum of the first slice start: one of the four lanes of a column holds its term, 1.
  const float scale2 = scale * kLog2E;
  const bool owns_sink = sinks && slice == 0;
  float m = owns_sink ? sinks[head] * kLog2E : -INFINITY, l = (owns_sink && g == 0) ? 1.f : 0.f;
  floatx4 acc[HDT];
#pragma unroll
  for (int i = 0; i < HDT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};

  // ---- One tile: 32 keys, in two halves of one page each.  Which key an operand's row stands for is free: row c of the
  // scores' u-th instruction is key 8 (c / 4) + 4 u + c % 4, so that a lane's eight probabilities are those of keys 8 g ... 8 g + 7
  // and the values that go with them are one load of 16 bytes.
  struct Tile {
    bf16x8 k[2][KS], v[HDT];
    unsigned mask;             // which of its keys are read (0: there is no such tile)
  };
  auto bits = [](int lo, int hi) -> unsigned {               // lo ... hi - 1 of 32 (lo < hi)
    return (~0u >> (32 - min(max(hi, 1), 32))) & (~0u << min(max(lo, 0), 31));
  };
  auto tile_key = [&](int tile) { return (KEPT && tile < n_kept) ? tile * 32 : first + (tile - n_kept) * 32; };
  // Where the 64 halves of 32 tiles from b0 on lie, a half to a lane: all their pages are one load.  A half that is not read
  // (its page may be gone) reads page 0.
  struct Places {
    unsigned mask;
    int slot;
    long base;               // bytes from the cache's first to the page's keys of this head
  };
  auto lookup = [&](int b0) -> Places {
    Places P;
    const int tile = b0 + lane / 2, kb = tile_key(tile), kept = min(keep_first, len) - kb;
    P.mask = KEPT && tile < n_kept ? bits(0, kept_end - kb) : bits(start - kb, len - kb) | (KEPT && kept > 0 ? bits(0, kept) : 0u);
    P.mask = tile < tile1 ? P.mask : 0u;
    const bool live = (P.mask >> (16 * (lane % 2))) & 0xFFFFu;
    unsigned left;
    const int index = (int)divided(live ? (unsigned)kb / 16 + lane % 2 : 0u, (unsigned)page16, page_magic, left);
    const int page = table[index];
    P.slot = (int)left * 16;
    P.base = (((long)(live ? page : 0) * 2 * KV + kvh) * block) * 2;
    return P;
  };
  const int k_lane = ((8 * (c / 4 % 2) + c % 4) * hd + 8 * g) * 2;       // bytes of this lane in a half's keys
  const int k_past = hd % 32 && g >= 2 ? -16 * g : 64 * (KS - 1);        // the last step: columns beyond the head read others (q is zero there)
  const int v_lane = (c * page_size + 8 * (g % 2)) * 2;                  // ... and in a page's values
  const int v_row = 32 * page_size;                                      // bytes from sixteen rows of values to the next
  auto fetch = [&](const Places& P, int i) -> Tile {         // the i-th of those tiles
    Tile T;
    T.mask = __builtin_amdgcn_readlane(P.mask, 2 * i);
    const char* kp[2];
    const char* vp[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned lo = __builtin_amdgcn_readlane((int)P.base, 2 * i + h);
      const long base = (long)((unsigned long)(unsigned)__builtin_amdgcn_readlane((int)(P.base >> 32), 2 * i + h) << 32 | lo);
      const int slot = __builtin_amdgcn_readlane(P.slot, 2 * i + h);
      kp[h] = reinterpret_cast<const char*>(cache) + base + slot * (2 * hd);
      vp[h] = reinterpret_cast<const char*>(cache) + base + 2 * KV * block + slot * 2;
    }
    __builtin_amdgcn_sched_barrier(0);
    const char* kl = (c < 8 ? kp[0] : kp[1]) + k_lane;
    const char* vl = (g < 2 ? vp[0] : vp[1]) + v_lane;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        T.k[u][ks] = *reinterpret_cast<const bf16x8*>(kl + 8 * u * hd + (hd % 32 && ks == KS - 1 ? k_past : 64 * ks));
    __builtin_amdgcn_sched_barrier(0);     // (keys first: the scores wait for no values)
#pragma unroll
    for (int r = 0; r < HDT; ++r) T.v[r] = *reinterpret_cast<const bf16x8*>(vl + (long)r * v_row);
    __builtin_amdgcn_sched_barrier(0);
    return T;
  };
  auto compute = [&](Tile& T, int tile) {
    floatx4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(T.k[u][ks], qb[ks], s[u], 0, 0, 0);
    }
    // ---- online softmax for this lane's head over its 8 keys, then the 4 lanes of the column
    float sc[8], tmax;
    const int far = BIASED ? len - 1 - tile_key(tile) - 8 * g : 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sc[e] = s[e / 4][e % 4] * scale2;
      if (BIASED) sc[e] -= slope * (float)(far - e);         // (a constant of the code: a model without slopes has none of it)
    }
    if (T.mask != ~0u) {                                     // first and last tiles: what is not read may hold anything
      const unsigned mine = T.mask >> (8 * g);
#pragma unroll
      for (int e = 0; e < 8; ++e) sc[e] = (mine >> e) & 1u ? sc[e] : -INFINITY;
      typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
      uint4_t keep;
#pragma unroll
      for (int d = 0; d < 4; ++d) keep[d] = ((mine >> (2 * d)) & 1u ? 0xFFFFu : 0u) | ((mine >> (2 * d + 1)) & 1u ? 0xFFFF0000u : 0u);
#pragma unroll
      for (int r = 0; r < HDT; ++r) T.v[r] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(uint4_t, T.v[r]) & keep);
    }
    tmax = sc[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) tmax = fmaxf(tmax, sc[e]);
    const float m_new = fmaxf(m, group4_max(tmax));        // finite: every tile holds a readable key
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    bf16x8 pb;
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bf16_t pr = (bf16_t)__builtin_amdgcn_exp2f(sc[e] - m_new);
      pb[e] = pr;
      psum += (float)pr;
    }
    l = l * alpha + psum;
    if (__builtin_amdgcn_ballot_w64(m_new > m)) {            // (after a few tiles the maximum rarely moves)
#pragma unroll
      for (int r = 0; r < HDT; ++r) acc[r] *= alpha;
    }
    m = m_new;
#pragma unroll
    for (int r = 0; r < HDT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(T.v[r], pb, acc[r], 0, 0, 0);
  };
  // While a tile is multiplied the next one's operands are on their way, in two buffers by name (a copy of one into the other
  // would wait for its loads).  Beyond the wave's last tile that one is asked for again.
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

  // ---- the waves' results meet in LDS; then a thread merges, in the order of the waves,
  // four elements of one head and writes them: the output itself where this workgroup had
  // all the keys, else the workgroup's partial result
  extern __shared__ __attribute__((aligned(16))) float red[];   // [waves][heads of the tile][hd + 4]
  constexpr int RS = hd + 4;                                 // row stride: 16-byte rows
  const int heads_here = min(16, G - ht * 16);
  if (head_ok) {
    float* mine = red + (wave * heads_here + c) * RS;
#pragma unroll
    for (int r = 0; r < HDT; ++r) *reinterpret_cast<floatx4*>(mine + 16 * r + 4 * g) = acc[r];
    if (g == 0) {
      mine[hd] = m;
      mine[hd + 1] = l;
    }
  }
  __syncthreads();
  const bool whole = wgs == 1;
  constexpr int CH = hd / 4;                                 // pieces of four elements in a head
  for (int idx = threadIdx.x; idx < heads_here * CH; idx += 64 * kDecodeWaves) {
    const int hc = idx / CH, d4 = (idx % CH) * 4;
    const float* col = red + hc * RS;
    float mj[kDecodeWaves], M = -INFINITY;
#pragma unroll
    for (int j = 0; j < kDecodeWaves; ++j) {
      mj[j] = col[j * heads_here * RS + hd];
      M = fmaxf(M, mj[j]);
    }
    const bool any = M != -INFINITY;                         // a workgroup beyond the last key has nothing
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
#pragma unroll
    for (int j = 0; j < kDecodeWaves; ++j) {
      const float* w = col + j * heads_here * RS;
      const float wj = any ? __builtin_amdgcn_exp2f(mj[j] - M) : 0.f;
      L += wj * w[hd + 1];
      v += wj * *reinterpret_cast<const floatx4*>(w + d4);
    }
    const int head_o = kvh * G + ht * 16 + hc;
    if (whole) {
      const float inv = 1.f / L;
      const floatx4 og = out_gate4(gate, t, head_o, d4);
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (bf16_t)(v[i] * inv * og[i]);
      *reinterpret_cast<bf16x4*>(final_out + (TILED ? rows_at(gate.side, t, head_o * hd + d4, H * hd)
                                                     : ((long)t * H + head_o) * hd + d4)) = o;
    } else {
      float* out = part + (((long)t * H + head_o) * wgs + place_wg) * (hd + 2);   // 8-byte rows
      *reinterpret_cast<floatx2*>(out + d4) = floatx2{v[0], v[1]};
      *reinterpret_cast<floatx2*>(out + d4 + 2) = floatx2{v[2], v[3]};
      if (d4 == 0) *reinterpret_cast<floatx2*>(out + hd) = floatx2{M * kLn2, L};
    }
  }
}

}  // namespace kllm
