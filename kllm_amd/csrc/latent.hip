// Attention through low-rank latents.  Per token one vector is cached for all heads: the
// normalised latent c [rank] followed by one rotated key part [dr].  A head's key is
// [W_uk,h c | rotated part] and its value W_uv,h c, so with the query's unrotated part folded
// through W_uk,h (q' = W_uk,h^T q, [rank]) the score is q' . c + q_rot . k_rot, the weighted
// sum over the keys is taken of c itself, and W_uv,h is applied once to that sum:
//
//   latent_kv_append   sums of W_dkv h -> RMS norm (weights) of the first rank, rotation of the
//                      last dr (halves paired), appended to the pages (one row of rank + dr a slot)
//   latent_query       sums of W_uq c_q -> per head [W_uk,h^T q_h | rotated q_h], rank + dr wide
//   attn_latent        one workgroup a (token, head): online softmax over 256 keys at a time,
//                      the values being the first rank elements of the cached rows; with a window
//                      the last `window` keys only (pages behind it may be gone)
//   latent_out         per head W_uv,h times the attended latent, times sigmoid of the gate's sums
//                      (one gate an element, or one a head)
//
// Scores, softmax, norms and rotation are 32-bit; the cached rows, the folded queries and the
// attended latents are stored in the compute type.
//
// A page holds its slots' rows [slot][rank + dr] and then the latents once more, transposed
// [rank][slot]: the weighted sum over the keys runs along the slots, and the matrix cores want
// the dimension that is summed over contiguous.  attn_latent has two kernels: one workgroup a
// (token, head) in 32-bit arithmetic for every size and type, and, in bfloat16 for ranks in
// steps of 16 and rows in steps of 8, one on the matrix cores (below).
#include <math.h>

#include <type_traits>
#include <stdint.h>

#include "common.hpp"
#include "kllm_kernels.h"

namespace kllm {

constexpr int kLatThreads = 256;
constexpr int kLatMaxRow = 1024;       // rank + dr of a cached row
constexpr int kLatMaxPer = kLatMaxRow / kLatThreads;

// A decode batch's launch is trips to memory in a row: position, span, a row's sums, weights and the rotation are asked for at once, with
// arguments that came with the launch; the page is the second trip.  PER * kLatThreads >= rank.  8 tokens of 512 + 64: 4.9 -> 3.6 us; 1,500 tokens
// 9.3 -> 7.7.
template <typename T, int PER>
__global__ __launch_bounds__(kLatThreads) void latent_kv_append_kernel(
    const int* __restrict__ positions, const int* __restrict__ span_of_token, const float* __restrict__ dkv, long in_stride, int rank, int dr,
    const float* __restrict__ weight, const int* __restrict__ block_table, int max_pages, int page_size, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int nsplit, long split_stride, float eps, T* __restrict__ cache) {
  __shared__ float red[16];
  const long t = blockIdx.x;
  int at = blockIdx.x;                        // (vector loads: scalar ones come one behind the other)
  asm volatile("" : "+v"(at));
  const int pos_v = positions[at], span_v = span_of_token[at];
  const int tid = threadIdx.x;
  const int row = rank + dr, half = dr / 2;
  const float* in = dkv + t * in_stride;
  float v[PER], w[PER], x[2][2], cs[2], sn[2];
#pragma unroll
  for (int q = 0; q < PER; ++q) v[q] = in[min(tid + q * kLatThreads, rank - 1)];
  asm volatile("" ::"s"(page_size), "s"(cos_t), "s"(sin_t), "s"(nsplit), "s"(split_stride), "s"(eps), "s"(cache));
#pragma unroll
  for (int q = 0; q < PER; ++q) w[q] = weight[min(tid + q * kLatThreads, rank - 1)];
#pragma unroll
  for (int q = 0; q < 2; ++q) {               // (up to 512 pairs)
    const int i = tid + q * kLatThreads;
    if (i < half) {
      x[q][0] = in[rank + i];
      x[q][1] = in[rank + half + i];
      cs[q] = cos_t[t * half + i];
      sn[q] = sin_t[t * half + i];
    }
  }
  const int pos = __builtin_amdgcn_readfirstlane(pos_v), span = __builtin_amdgcn_readfirstlane(span_v);
  const int page_in = pos / page_size, slot = pos - page_in * page_size;
  const long entry = (long)span * max_pages + page_in;
  const int page_v = block_table[entry];
  for (int s = 1; s < nsplit; ++s) {
#pragma unroll
    for (int q = 0; q < PER; ++q) v[q] += in[s * split_stride + min(tid + q * kLatThreads, rank - 1)];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = tid + q * kLatThreads;
      if (i < half) {
        x[q][0] += in[s * split_stride + rank + i];
        x[q][1] += in[s * split_stride + rank + half + i];
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < PER; ++q)
    if (tid + q * kLatThreads < rank) ss = fmaf(v[q], v[q], ss);
  const float rstd = 1.f / sqrtf(block_sum(ss, red) / (float)rank + eps);
  const long page_elems = (long)page_size * (row + rank), page = page_v;
  T* dst = cache + page * page_elems + (long)slot * row;
  T* dst_t = cache + page * page_elems + (long)page_size * row + slot;     // [rank][slot]
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int i = tid + q * kLatThreads;
    if (i < rank) {
      const T c = from_f32<T>(v[q] * rstd * w[q]);
      dst[i] = c;
      dst_t[(long)i * page_size] = c;
    }
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = tid + q * kLatThreads;
    if (i < half) {
      dst[rank + i] = from_f32<T>(x[q][0] * cs[q] - x[q][1] * sn[q]);
      dst[rank + half + i] = from_f32<T>(x[q][1] * cs[q] + x[q][0] * sn[q]);
    }
  }
}

// out [n][r] = N(in row's r elements) * weight, the rows of `in` in_stride apart; one workgroup a row.
// PER > 0: rows of up to PER * kLatThreads elements, which a thread keeps in registers, so that its
// loads (a slice's all together) are one trip to memory each; rows of 1,536 with eight numbers a thread instead of sixteen: 8 tokens 5.1 -> 3.5 us,
// 1,500 tokens 9.0 -> 5.3.
template <typename T, int PER>
__global__ __launch_bounds__(kLatThreads) void latent_norm_kernel(const float* __restrict__ in, const float* __restrict__ weight, long in_stride, int r,
                                                                  int nsplit, T* __restrict__ out, float eps, long split_stride) {
  __shared__ float red[16];
  const long t = blockIdx.x;
  const int tid = threadIdx.x;
  const float* src = in + t * in_stride;
  float ss = 0.f;
  if constexpr (PER > 0) {
    float v[PER], w[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = src[min(tid + kLatThreads * j, r - 1)];
    asm volatile("" ::"s"(split_stride));
#pragma unroll
    for (int j = 0; j < PER; ++j) w[j] = weight[min(tid + kLatThreads * j, r - 1)];
    for (int s = 1; s < nsplit; ++s)
#pragma unroll
      for (int j = 0; j < PER; ++j) v[j] += src[s * split_stride + min(tid + kLatThreads * j, r - 1)];
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (tid + kLatThreads * j < r) ss = fmaf(v[j], v[j], ss);
    const float rstd = 1.f / sqrtf(block_sum(ss, red) / (float)r + eps);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (tid + kLatThreads * j < r) out[t * r + tid + kLatThreads * j] = from_f32<T>(v[j] * rstd * w[j]);
    return;
  }
  for (int i = tid; i < r; i += kLatThreads) {
    float v = 0.f;
    for (int s = 0; s < nsplit; ++s) v += src[s * split_stride + i];
    ss = fmaf(v, v, ss);
  }
  const float rstd = 1.f / sqrtf(block_sum(ss, red) / (float)r + eps);
  for (int i = tid; i < r; i += kLatThreads) {
    float v = 0.f;
    for (int s = 0; s < nsplit; ++s) v += src[s * split_stride + i];
    out[t * r + i] = from_f32<T>(v * rstd * weight[i]);
  }
}

// q: [nsplit][n][H * (d + dr)], a head laid out [d unrotated | dr rotated]; w_uk [H * d][rank].
template <typename T>
__global__ __launch_bounds__(kLatThreads) void latent_query_kernel(
    const float* __restrict__ q, int nsplit, long split_stride, const T* __restrict__ w_uk,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, T* __restrict__ out, int H, int d, int dr,
    int rank) {
  extern __shared__ float qh[];          // [d + dr]
  const long t = blockIdx.x;
  const int h = blockIdx.y, tid = threadIdx.x;
  const int hw = d + dr, half = dr / 2;
  const float* in = q + (t * H + h) * hw;
  for (int i = tid; i < hw; i += kLatThreads) {
    float v = 0.f;
    for (int s = 0; s < nsplit; ++s) v += in[s * split_stride + i];
    qh[i] = v;
  }
  __syncthreads();
  T* dst = out + (t * H + h) * (rank + dr);
  const T* w = w_uk + (long)h * d * rank;
  for (int r = tid; r < rank; r += kLatThreads) {
    float acc = 0.f;
    for (int i = 0; i < d; ++i) acc = fmaf(qh[i], to_f32(w[(long)i * rank + r]), acc);
    dst[r] = from_f32<T>(acc);
  }
  for (int i = tid; i < half; i += kLatThreads) {
    const float a = qh[d + i], b = qh[d + half + i];
    const float c = cos_t[t * half + i], sn = sin_t[t * half + i];
    dst[rank + i] = from_f32<T>(a * c - b * sn);
    dst[rank + half + i] = from_f32<T>(b * c + a * sn);
  }
}

template <typename T>
__global__ __launch_bounds__(kLatThreads) void attn_latent_kernel(
    const T* __restrict__ q, T* __restrict__ out, const T* __restrict__ cache, const int* __restrict__ positions,
    const int* __restrict__ span_of_token, const int* __restrict__ block_table, int max_pages, int page_size, int H,
    int row, int rank, float scale, int window) {
  __shared__ float qs[kLatMaxRow];
  __shared__ float ps[kLatThreads];
  __shared__ float red[16];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const long page_elems = (long)page_size * (row + rank);
  const int len = positions[t] + 1;
  const int lo = first_key(len - 1, window, 0);
  const int* table = block_table + (long)span_of_token[t] * max_pages;
  const T* qrow = q + ((long)t * H + h) * row;
  for (int i = tid; i < row; i += kLatThreads) qs[i] = to_f32(qrow[i]);
  __syncthreads();
  float m = -INFINITY, l = 0.f;
  float acc[kLatMaxPer];
#pragma unroll
  for (int c = 0; c < kLatMaxPer; ++c) acc[c] = 0.f;
  for (int base = lo; base < len; base += kLatThreads) {
    const int key = base + tid;
    float s = -INFINITY;
    if (key < len) {
      const T* krow = cache + (long)table[key / page_size] * page_elems + (long)(key % page_size) * row;
      float dot = 0.f;
      for (int i = 0; i < row; ++i) dot = fmaf(qs[i], to_f32(krow[i]), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, block_max(s, red));
    const float alpha = expf(m - m_new);
    const float p = (s == -INFINITY) ? 0.f : expf(s - m_new);
    ps[tid] = p;
    l = l * alpha + block_sum(p, red);       // its barriers also publish ps
    m = m_new;
    const int nk = min(kLatThreads, len - base);
#pragma unroll
    for (int c = 0; c < kLatMaxPer; ++c) {
      const int e = tid + c * kLatThreads;
      acc[c] *= alpha;
      if (e < rank) {
        float a = acc[c];
        int pg = -1;
        const T* prow = nullptr;
        for (int k = 0; k < nk; ++k) {
          const int kk = base + k;
          if (kk / page_size != pg) {
            pg = kk / page_size;
            prow = cache + (long)table[pg] * page_elems;
          }
          a = fmaf(ps[k], to_f32(prow[(long)(kk % page_size) * row + e]), a);
        }
        acc[c] = a;
      }
    }
    __syncthreads();                         // ps is rewritten by the next round
  }
#pragma unroll
  for (int c = 0; c < kLatMaxPer; ++c) {
    const int e = tid + c * kLatThreads;
    if (e < rank) out[((long)t * H + h) * rank + e] = from_f32<T>(acc[c] / l);
  }
}

// attn_latent on the matrix cores (bfloat16).  A workgroup takes one token, up to 16 heads and, round by round, 128 of the token's
// keys.  All heads read the same keys, so the 16 heads are the columns of one product:
// MFMA 16x16x32 (lane l: g = l/16, c = l%16): A[c][8g..8g+7], B[8g..8g+7][c], D[4g+i][c].
// Scores: each of the four waves takes a tile of 32 keys, A = 16 of them x 32 elements of their rows (one row per lane, straight from the page),
// B = the folded queries of the 16 heads.  Which key stands in which row is free: key 8 (c / 4) + 4 u + c % 4 in row c of the u-th of two
// instructions, so that a lane's probabilities are those of eight neighbouring keys.  They meet in LDS (the heads' maxima first), and each
// wave takes a quarter of the weighted sum's elements for all four tiles: A = latents [element c][8 keys], 16 bytes from the transposed copy.
//
// What bounds a decode step's launch are its trips to memory (position and span; pages; rows and latents, all of a round asked for
// at once) and its code, which is read cold.  A wave that keeps all elements for its own keys needs four times the accumulators and
// a merge of them in LDS that leaves a CU one workgroup: 28 KB of code, 25 us for 8 tokens, 32 heads and 1,400 keys with rank 512 in 32 slices, most of them
// empty but writing their zeros; so 14, of which the rows and latents, 24 MB, take five at the rate of a large read.
// NR: 16-element pieces of the latent, KS: steps of 32 over a row that a lane asks for at once (0: four at a time, for rows longer
// than the built sizes).  The queries lie in LDS: in registers, with the round's keys and latents there, they were spilt.
constexpr int kLatWaves = 4;

template <int NR, int KS>
__global__ __launch_bounds__(64 * kLatWaves) void attn_latent_mfma_kernel(
    const bf16_t* __restrict__ cache, const int* __restrict__ positions, const int* __restrict__ span_of_token,
    const int* __restrict__ block_table, const bf16_t* __restrict__ q, int max_pages, int page16, int H, int row, int rank, unsigned page_magic,
    float scale, int window, int nslices, bf16_t* __restrict__ out, float* __restrict__ part) {
  constexpr int PER = NR / kLatWaves;           // pieces of a wave: wave, wave + 4, ...
  // Steps that lie in every row of the instance (row >= rank, and the launch's limits): their places are constants in the loads.  A place
  // worked out for every step spilt 19 registers with rows of 640 (1 / 8 / 32 tokens at 1,400 keys 14.5 / 17.3 / 32.2 us, so 12.9 / 16.5 / 29.8).
  constexpr int SURE = KS == 0 ? 0 : KS == 20 ? 18 : NR == 32 ? 8 : NR == 16 ? 4 : 0;
  constexpr int PLD = 32 * kLatWaves + 8;       // probabilities of a head's 128 keys in LDS, and a shift of banks
  __shared__ __attribute__((aligned(16))) bf16_t probs[2][16 * PLD];
  constexpr int QLD = (KS > 0 ? 32 * KS : kLatMaxRow) + 8;
  __shared__ __attribute__((aligned(16))) bf16_t queries[16 * QLD];
  __shared__ float meet[2][kLatWaves][16];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 16, c = lane % 16;
  const int t = blockIdx.x, h0 = blockIdx.y * 16, slice = blockIdx.z;
  int at = t;
  asm volatile("" : "+v"(at));                  // (vector loads, as in decode attention: they go out together)
  const int pos_v = positions[at], span_v = span_of_token[at];
  asm volatile("" ::"s"(rank), "s"(page_magic), "s"(scale), "s"(window), "s"(nslices), "s"(out), "s"(part));
  const int page_size = 16 * page16;
  const int head = min(h0 + c, H - 1);
  const bool head_ok = h0 + c < H;
  int len = __builtin_amdgcn_readfirstlane(pos_v) + 1, span = __builtin_amdgcn_readfirstlane(span_v);
  asm volatile("" : "+s"(len), "+s"(span));
  const int lo = first_key(len - 1, window, 0);        // the first key that is read
  const int tile0 = lo / 32, rounds = (len - 32 * tile0 + 127) / 128;
  float* prow = part + (((long)t * H + head) * nslices + slice) * (rank + 2);     // (of several slices) rows of rank + 2 floats
  if (slice >= rounds) {                               // no keys: a maximum of -inf, and the merge reads no more of it
    if (wave == 0 && g == 0 && head_ok) *reinterpret_cast<floatx2*>(prow + rank) = floatx2{-INFINITY, 0.f};
    return;
  }
  const int* table = block_table + (long)span * max_pages;
  const long page_bytes = 2L * page_size * (row + rank);
  const float scale2 = scale * kLog2E;
  auto bits = [](int from, int to) -> unsigned {       // from ... to - 1 of 32
    return to <= 0 || from >= 32 ? 0u : (~0u >> (32 - min(to, 32))) & (~0u << max(from, 0));
  };
  // Where the 64 halves of eight rounds from r0 on lie, a half (16 keys in one page) to a lane: their pages are one load.
  // A half that is not read (its page may be gone) reads page 0.
  struct Places {
    unsigned mask;                              // of the half's tile: which keys are read
    int slot;
    long base;                                  // bytes from the cache's first to the half's page
  };
  auto lookup = [&](int r0) -> Places {
    Places P;
    const int kb = 32 * (tile0 + 4 * (r0 + lane / 8 * nslices) + lane % 8 / 2);
    P.mask = bits(lo - kb, len - kb);
    const bool live = (P.mask >> (16 * (lane % 2))) & 0xFFFFu;
    unsigned left;
    const int index = (int)divided(live ? (unsigned)kb / 16 + lane % 2 : 0u, (unsigned)page16, page_magic, left);
    P.slot = live ? (int)left * 16 : -1;
    P.base = table[index];
    return P;
  };
  auto placed = [&](Places P) -> Places {              // once the pages are there
    P.base = (long)(P.slot >= 0 ? (int)P.base : 0) * page_bytes;
    P.slot = max(P.slot, 0);
    return P;
  };
  auto half_at = [&](const Places& P, int i) {
    const unsigned low = __builtin_amdgcn_readlane((int)P.base, i);
    return reinterpret_cast<const char*>(cache) +
           (long)((unsigned long)(unsigned)__builtin_amdgcn_readlane((int)(P.base >> 32), i) << 32 | low);
  };
  auto slot_at = [&](const Places& P, int i) { return __builtin_amdgcn_readlane(P.slot, i); };
  auto mask_at = [&](const Places& P, int i) -> unsigned { return __builtin_amdgcn_readlane((int)P.mask, i); };
  // A tile without keys reads the round's first one again: its scores are masked and its sums left out.
  auto key_row = [&](const Places& P, int i) {         // this lane's row of the wave's tile of the i-th round
    const int j = 8 * i + (mask_at(P, 8 * i + 2 * wave) ? 2 * wave : 0);
    const char* k0 = half_at(P, j) + (long)slot_at(P, j) * (2 * row);
    const char* k1 = half_at(P, j + 1) + (long)slot_at(P, j + 1) * (2 * row);
    return (c < 8 ? k0 : k1) + ((8 * (c / 4 % 2) + c % 4) * row + 8 * g) * 2;
  };
  auto k_at = [&](const char* kl, int kk, int u) {
    return *reinterpret_cast<const bf16x8*>(kl + 8 * u * row + (kk < SURE || 32 * kk + 8 * g < row ? 64 * kk : -16 * g));
  };
  struct Values {
    bf16x8 v[PER];
  };
  auto v_fetch = [&](const Places& P, int i, int w) -> Values {       // tile w of the i-th round
    Values V;
    const int j = 8 * i + (mask_at(P, 8 * i + 2 * w) ? 2 * w : 0);
    const char* v0 = half_at(P, j) + 2L * page_size * row + 2 * slot_at(P, j);
    const char* v1 = half_at(P, j + 1) + 2L * page_size * row + 2 * slot_at(P, j + 1);
    const char* vl = (g < 2 ? v0 : v1) + ((16 * wave + c) * page_size + 8 * (g % 2)) * 2;
#pragma unroll
    for (int r = 0; r < PER; ++r)
      V.v[r] = *reinterpret_cast<const bf16x8*>(vl + (16 * (4 * r + wave) < rank ? 128L * r * page_size : -32L * wave * page_size));
    return V;
  };

  Places first = lookup(slice);
  // The heads' queries go to LDS, zeros behind a row up to whole steps (there a key's row brings another piece of itself): asked for
  // behind the pages, written once the first keys are on their way.
  const int steps = KS > 0 ? KS : (row + 31) / 32;
  auto q_load = [&](int i) {
    const int h = i / (4 * steps), d0 = 8 * (i % (4 * steps));
    return *reinterpret_cast<const bf16x8*>(q + ((long)t * H + min(h0 + h, H - 1)) * row + (d0 < row ? d0 : 0));
  };
  auto q_store = [&](int i, bf16x8 v) {
    const int h = i / (4 * steps), d0 = 8 * (i % (4 * steps));
    if (d0 >= row) v = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    *reinterpret_cast<bf16x8*>(&queries[h * QLD + d0]) = v;
  };
  auto q_at = [&](int kk) { return *reinterpret_cast<const bf16x8*>(&queries[c * QLD + 32 * kk + 8 * g]); };
  constexpr int QN = KS > 0 ? (64 * KS + 64 * kLatWaves - 1) / (64 * kLatWaves) : 1;
  bf16x8 qv[QN];
  if constexpr (KS > 0) {
#pragma unroll
    for (int j = 0; j < QN; ++j) qv[j] = q_load(min((int)threadIdx.x + 64 * kLatWaves * j, 64 * KS - 1));
    __builtin_amdgcn_sched_barrier(0);
  }

  float m = -INFINITY, l = 0.f;
  floatx4 acc[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};
  int parity = 0;
  for (int r0 = slice; r0 < rounds; r0 += 8 * nslices) {
    if (r0 != slice) first = lookup(r0);
    const Places P = placed(first);
    bf16x8 kr[KS > 0 ? KS : 1][2];
    auto k_fetch = [&](int i) {
      const char* kl = key_row(P, i);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int u = 0; u < 2; ++u) kr[kk][u] = k_at(kl, kk, u);
      __builtin_amdgcn_sched_barrier(0);
    };
    k_fetch(0);
    if (r0 == slice) {
      if constexpr (KS > 0) {
#pragma unroll
        for (int j = 0; j < QN; ++j) q_store(min((int)threadIdx.x + 64 * kLatWaves * j, 64 * KS - 1), qv[j]);
      } else {
        for (int i = threadIdx.x; i < 64 * steps; i += 64 * kLatWaves) q_store(i, q_load(i));
      }
      // (a wait for what goes to LDS and for nothing else, written out: the keys stay on their way)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
#pragma unroll 1
    for (int i = 0; i < 8 && r0 + i * nslices < rounds; ++i, parity ^= 1) {
      Values V[kLatWaves];
#pragma unroll
      for (int w = 0; w < kLatWaves; ++w) V[w] = v_fetch(P, i, w);
      __builtin_amdgcn_sched_barrier(0);
      floatx4 s[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
      if constexpr (KS > 0) {
        constexpr int QB = KS % 6 == 0 ? 6 : 4;        // pieces of the query, a group ahead of the products
        static_assert(KS % QB == 0, "whole groups of steps");
        bf16x8 qb[2][QB];
#pragma unroll
        for (int kk = 0; kk < QB; ++kk) qb[0][kk] = q_at(kk);
#pragma unroll
        for (int k0 = 0; k0 < KS; k0 += QB) {
#pragma unroll
          for (int kk = 0; kk < QB; ++kk)
            if (k0 + QB < KS) qb[(k0 / QB + 1) % 2][kk] = q_at(k0 + QB + kk);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk < QB; ++kk)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[k0 + kk][u], qb[k0 / QB % 2][kk], s[u], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i < 7 && r0 + (i + 1) * nslices < rounds) k_fetch(i + 1);
      } else {
        const char* kl = key_row(P, i);
        for (int k0 = 0; k0 < steps; k0 += 4) {
          bf16x8 kv[4][2];
#pragma unroll
          for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int u = 0; u < 2; ++u) kv[kk][u] = k_at(kl, min(k0 + kk, steps - 1), u);
#pragma unroll
          for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              if (k0 + kk < steps) s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv[kk][u], q_at(k0 + kk), s[u], 0, 0, 0);
        }
      }
      // ---- online softmax, in units of log2(e): the heads' maxima over the round's four tiles first
      const unsigned mine = mask_at(P, 8 * i + 2 * wave) >> (8 * g);
      float sc[8], tmax = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sc[e] = (mine >> e) & 1u ? s[e / 4][e % 4] * scale2 : -INFINITY;
        tmax = fmaxf(tmax, sc[e]);
      }
      tmax = group4_max(tmax);
      if (g == 0) meet[parity][wave][c] = tmax;
      __syncthreads();
      float m_new = m;
#pragma unroll
      for (int w = 0; w < kLatWaves; ++w) m_new = fmaxf(m_new, meet[parity][w][c]);     // finite: every round holds a key that is read
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      bf16x8 pb;
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pb[e] = (bf16_t)__builtin_amdgcn_exp2f(sc[e] - m_new);
        psum += (float)pb[e];
      }
      *reinterpret_cast<bf16x8*>(&probs[parity][c * PLD + 32 * wave + 8 * g]) = pb;
      l = l * alpha + psum;
      if (__builtin_amdgcn_ballot_w64(m_new > m)) {
#pragma unroll
        for (int r = 0; r < PER; ++r) acc[r] *= alpha;
      }
      m = m_new;
      __syncthreads();
      // ---- the weighted sum of the latents: slots of keys that are not read may hold anything
#pragma unroll
      for (int w = 0; w < kLatWaves; ++w) {
        const unsigned mask = mask_at(P, 8 * i + 2 * w);
        if (mask != ~0u) {
          typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
          const unsigned own = mask >> (8 * g);
          uint4_t keep;
#pragma unroll
          for (int d = 0; d < 4; ++d) keep[d] = ((own >> (2 * d)) & 1u ? 0xFFFFu : 0u) | ((own >> (2 * d + 1)) & 1u ? 0xFFFF0000u : 0u);
#pragma unroll
          for (int r = 0; r < PER; ++r) V[w].v[r] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(uint4_t, V[w].v[r]) & keep);
        }
        const bf16x8 pw = *reinterpret_cast<const bf16x8*>(&probs[parity][c * PLD + 32 * w + 8 * g]);
#pragma unroll
        for (int r = 0; r < PER; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(V[w].v[r], pw, acc[r], 0, 0, 0);
      }
    }
  }
  l = group4_sum(l);
  if (g == 0) meet[parity][wave][c] = l;
  __syncthreads();
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < kLatWaves; ++w) L += meet[parity][w][c];
  if (!head_ok) return;
  // of a slice the sums as they are, with its maximum (in units of log2(e)) and its sum of probabilities
  const float inv = 1.f / L;
  bf16_t* orow = out + ((long)t * H + head) * rank;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int r = 4 * j + wave;
    if (16 * r >= rank) continue;
    if (nslices > 1) {                                       // (rows are 8-byte aligned)
      *reinterpret_cast<floatx2*>(prow + 16 * r + 4 * g) = floatx2{acc[j][0], acc[j][1]};
      *reinterpret_cast<floatx2*>(prow + 16 * r + 4 * g + 2) = floatx2{acc[j][2], acc[j][3]};
    } else {
      *reinterpret_cast<bf16x4*>(orow + 16 * r + 4 * g) =
          bf16x4{(bf16_t)(acc[j][0] * inv), (bf16_t)(acc[j][1] * inv), (bf16_t)(acc[j][2] * inv), (bf16_t)(acc[j][3] * inv)};
    }
  }
  if (nslices > 1 && wave == 0 && g == 0) *reinterpret_cast<floatx2*>(prow + rank) = floatx2{m, L};
}

// The same for steps of many tokens: a workgroup takes four consecutive tokens of the step and up
// to 16 heads, one token a wave.  Tokens of one request read the same keys: a tile of 32 keys
// (their rows, and their latents with the keys side by side) goes through LDS once for the
// four, which cuts the traffic between L2 and the CUs to a quarter.  Where the four tokens
// belong to several requests, the requests take their turns.  No merge: a wave has all keys
// of its token.  LDS: rows [32][row + 8], latents [rank][32 + 4] (padded against bank conflicts).
template <int NR, int KS>
__global__ __launch_bounds__(64 * kLatWaves) void attn_latent_block_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
    const int* __restrict__ positions, const int* __restrict__ span_of_token, const int* __restrict__ block_table,
    int max_pages, int page_size, unsigned page_magic, int n, int H, int row, int rank, float scale, int window, int redo) {
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_tiles[];
  // page of a key without a division: page_magic = ceil(2^35 / page_size) from the host, exact for
  // keys below 2^24 and pages of up to 2,048 slots (checked at the launch)
  auto page_index = [&](int key) { return (int)(__umulhi((unsigned)key, page_magic) >> 3); };
  const int KLD = row + 8, VLD = 36;
  bf16_t* ks = lat_tiles;                      // [32][KLD]
  bf16_t* vs = lat_tiles + 32 * KLD;           // [rank][VLD]
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int g = lane / 16, c = lane % 16;
  // later tokens of a prompt read more keys: the workgroups with the most to do start first
  const int t_first = (gridDim.x - 1 - blockIdx.x) * kLatWaves, h0 = blockIdx.y * 16;
  const int t = min(t_first + wave, n - 1);
  const bool token_ok = t_first + wave < n;
  const int head = min(h0 + c, H - 1);
  const bool head_ok = h0 + c < H;
  // behind attn_latent_columns_kernel: only where that left a column to be done
  if (redo && !__syncthreads_or(token_ok && head_ok && isnan((float)out[((long)t * H + head) * rank]))) return;
  const int my_span = span_of_token[t];
  const int len = positions[t] + 1;
  const int lo = first_key(len - 1, window, 0);
  const long page_elems = (long)page_size * (row + rank);
  const int ksteps = (row + 31) / 32, nr = rank / 16;
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16_t* qrow = q + ((long)t * H + head) * row;
  const int rows_here = min(kLatWaves, n - t_first);
  bf16x8 qreg[KS > 0 ? KS : 1];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) {
    const int d0 = 32 * kk + 8 * g;
    qreg[kk] = (d0 < row && head_ok) ? *reinterpret_cast<const bf16x8*>(qrow + d0) : zero8;
  }

  float m = -INFINITY, l = 0.f;
  floatx4 acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};

  for (int first = 0; first < rows_here;) {
    const int span = span_of_token[t_first + first];
    int last = first;
    while (last + 1 < rows_here && span_of_token[t_first + last + 1] == span) ++last;
    const int group_len = positions[t_first + last] + 1;      // the group's last token reads the most keys
    const int group_lo = first_key(positions[t_first + first], window, 0);   // ... and its first the earliest (pages before it may be gone)
    const bool mine = token_ok && wave >= first && wave <= last;
    const int* table = block_table + (long)span * max_pages;
    // ---- a tile's way into LDS, 16 bytes at a time.  Thread tid moves pieces tid % 8, + 8, ... of key row
    // tid / 8, and 8 keys (part tid % 4) of elements tid / 4, + 64, ...: the same places in every tile.
    // For the built row sizes the pieces of the NEXT tile are asked for before the products of this
    // one and wait in registers meanwhile, their pages having been looked up a tile earlier, and no
    // load has a branch around it: a half (16 keys, in one page) that nobody reads takes page 0;
    // its scores are masked (a row is one key's alone), its latents replaced by zeros.
    constexpr int KP = KS > 0 ? KS / 2 : 1, VP = NR / 4;      // pieces a thread: of 32 rows of up to 32 KS, of 16 NR elements
    struct Stage {
      bf16x8 k[KP], v[VP];
    };
    struct Halves {
      int page[2];
    };
    const int row8 = row / 8;
    const int kr = tid / 8, kc = tid % 8, ve = tid / 4, vpart = tid % 4;
    auto half_live = [&](int k0) { return k0 < group_len && k0 + 16 > group_lo; };
    auto lookup = [&](int kb) -> Halves {
      Halves P;
#pragma unroll
      for (int u = 0; u < 2; ++u) P.page[u] = table[half_live(kb + 16 * u) ? page_index(kb + 16 * u) : 0];
      return P;
    };
    auto place = [&](const Halves& P, int k0, int u) -> const bf16_t* {      // the half's first row in its page
      const bool live = half_live(k0);
      return cache + (long)(live ? (u ? P.page[1] : P.page[0]) : 0) * page_elems;
    };
    auto slot_of = [&](int k0) { return half_live(k0) ? k0 - page_index(k0) * page_size : 0; };
    auto k_load = [&](const bf16_t* rows, int m) -> bf16x8 {
      const int piece = kc + 8 * m;
      return *reinterpret_cast<const bf16x8*>(rows + 8 * (piece < row8 ? piece : 0));
    };
    auto v_load = [&](const bf16_t* cols, int m) -> bf16x8 {
      return *reinterpret_cast<const bf16x8*>(cols + (long)min(ve + 64 * m, rank - 1) * page_size);
    };
    auto k_rows = [&](const Halves& P, int kb) {
      const int u = kr / 16, k0 = kb + 16 * u;
      return place(P, k0, u) + (long)(slot_of(k0) + kr % 16) * row;
    };
    auto v_cols = [&](const Halves& P, int kb) {
      const int u = vpart / 2, k0 = kb + 16 * u;
      return place(P, k0, u) + (long)page_size * row + slot_of(k0) + 8 * (vpart % 2);
    };
    auto k_store = [&](int m, const bf16x8& v) {
      const int piece = kc + 8 * m;
      if (piece < row8) *reinterpret_cast<bf16x8*>(ks + kr * KLD + 8 * piece) = v;
    };
    auto v_store = [&](int m, bf16x8 v, int kb) {
      if (ve + 64 * m >= rank) return;
      if (kb < group_lo || kb + 32 > group_len) {             // slots that may hold anything
        const int key = kb + 8 * vpart;
        const bool live = half_live(kb + 16 * (vpart / 2));
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (live && key + j < group_len) ? v[j] : (bf16_t)0.f;
      }
      bf16_t* dst = vs + (ve + 64 * m) * VLD + 8 * vpart;     // 8-byte aligned
      *reinterpret_cast<bf16x4*>(dst) = bf16x4{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<bf16x4*>(dst + 4) = bf16x4{v[4], v[5], v[6], v[7]};
    };
    auto fetch = [&](int kb, const Halves& P) -> Stage {
      Stage T;
      const bf16_t *kp = k_rows(P, kb), *vp = v_cols(P, kb);
#pragma unroll
      for (int m = 0; m < KP; ++m) T.k[m] = k_load(kp, m);
#pragma unroll
      for (int m = 0; m < VP; ++m) T.v[m] = v_load(vp, m);
      return T;
    };
    Stage st;
    Halves pages;
    const int kb0 = group_lo / 32 * 32;
    if constexpr (KS > 0) {
      pages = lookup(kb0);
      st = fetch(kb0, pages);
      pages = lookup(kb0 + 32);
    }
    for (int kb = kb0; kb < group_len; kb += 32) {
      __syncthreads();                                        // the tile before this one has been read
      if constexpr (KS > 0) {
#pragma unroll
        for (int m = 0; m < KP; ++m) k_store(m, st.k[m]);
#pragma unroll
        for (int m = 0; m < VP; ++m) v_store(m, st.v[m], kb);
      } else {
        pages = lookup(kb);
        const bf16_t *kp = k_rows(pages, kb), *vp = v_cols(pages, kb);
        for (int m = 0; 8 * m < row8; ++m) k_store(m, k_load(kp, m));
        for (int m = 0; 64 * m < rank; ++m) v_store(m, v_load(vp, m), kb);
      }
      __syncthreads();
      if constexpr (KS > 0) {                                 // (beyond the last tile: a valid address, dropped)
        st = fetch(kb + 32, pages);
        pages = lookup(kb + 64);
      }
      if (!mine || kb >= len || kb + 32 <= lo) continue;
      // ---- scores
      floatx4 s[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
      auto score_step = [&](int kk, const bf16x8& qb) {
        const int d0 = 32 * kk + 8 * g;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const bf16x8 a = d0 < row ? *reinterpret_cast<const bf16x8*>(ks + (16 * u + c) * KLD + d0) : zero8;
          s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qb, s[u], 0, 0, 0);
        }
      };
      if constexpr (KS > 0) {
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
          if (kk < ksteps) score_step(kk, qreg[kk]);
      } else {
        for (int kk = 0; kk < ksteps; ++kk) {
          const int d0 = 32 * kk + 8 * g;
          score_step(kk, (d0 < row && head_ok) ? *reinterpret_cast<const bf16x8*>(qrow + d0) : zero8);
        }
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kb + 16 * u + 4 * g + i;
          s[u][i] = (key < len && key >= lo) ? s[u][i] * scale : -INFINITY;
          tmax = fmaxf(tmax, s[u][i]);
        }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, kWave));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
      const float m_new = fmaxf(m, tmax);                    // finite: the tile holds a key of this token
      const float alpha = expf(m - m_new);
      bf16x8 pb;
      float psum = 0.f;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = (s[u][i] == -INFINITY) ? 0.f : expf(s[u][i] - m_new);
          const bf16_t pr = (bf16_t)p;
          pb[4 * u + i] = pr;
          psum += (float)pr;
        }
      l = l * alpha + psum;
      m = m_new;
      // ---- the weighted sum of the latents (keys beyond this token's last: probability 0, and
      // what LDS holds of them is another token's key or zero, never anything else)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        if (r < nr) {
          acc[r] *= alpha;
          const bf16_t* vrow = vs + (16 * r + c) * VLD + 4 * g;
          const bf16x4 lo = *reinterpret_cast<const bf16x4*>(vrow);
          const bf16x4 hi = *reinterpret_cast<const bf16x4*>(vrow + 16);
          const bf16x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb, acc[r], 0, 0, 0);
        }
      }
    }
    first = last + 1;
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  if (!token_ok || !head_ok) return;
  const float inv = 1.f / l;
  bf16_t* orow = out + ((long)t * H + head) * rank;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r < nr) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(acc[r][i] * inv);
      *reinterpret_cast<bf16x4*>(orow + 16 * r + 4 * g) = v;
    }
  }
}

// The same for long steps of the common sizes (rank and rows in steps of 32): the (token, head) pairs of a
// step in a row are columns, 128 to a workgroup and 32 to a wave, and the products are MFMA 32x32x16
// (lane l: g = l/32, c = l%32: A[c][8g..8g+7], B[8g..8g+7][c], D[8(i/4) + 4g + i%4][c]).  Scores S^T =
// K Q^T: A = 32 keys x 16 of their rows from LDS, row r of it the key r with bits 2 and 3 exchanged, B = the columns' folded
// queries, which stay in registers; a lane holds 16 scores of one column, lane ^ 32 the other 16: 8u + j that of key 16u + 8g + j.
// Weighted sum O^T += C^T P^T: the 16 slots of MFMA u are those keys, A = latents [element c][eight neighbouring keys], one read of 16 bytes.
//
// A tile of 32 keys (rows, then latents with the keys side by side) goes from the pages straight into one of
// two LDS buffers (global loads that write LDS: 16 bytes a lane, a wave's 64 pieces in a row), the
// next tile's while this one is multiplied, a load behind every two products of the scores: with a wave to a SIMD whatever is not a product stands in
// line with them, and the loads all at once in front of the first reads from LDS kept those waiting.  Reads of 8 bytes and loads in
// front -> now, us: 1,500 tokens of 32 heads, rank 512 156 -> 136, 700 82 -> 73, 4,000 of 16 heads 383 -> 333, 1,500 of 16 heads, rank 256 93 -> 85; slower where
// a request has one tile, behind which a second is asked for that nobody reads: 50 prompts of 30 tokens of 32 heads, rank 512 63.5 -> 64.1, of 16 38.8 -> 40.2,
// rank 256 23.1 -> 24.2 (loads around which the tile's last turn jumps: 12 % slower elsewhere).  A wave cannot pad what it writes this way, so the 16-byte
// pieces of a row change places: piece p of key row k lies at p ^ (k & row_mask), piece p of
// element e's 32 keys at p ^ (e/4 % 4), which spreads a read over the banks.
//
// The accumulators fill the matrix unit's own registers, and the query's pieces most of the others: there
// is no room to bring an output to a new maximum.  Probabilities are taken relative to the largest score
// of the column's first tile instead, which is exact as long as no later score is more than kLatRange
// binary orders above it (32-bit and bfloat16 numbers have the same exponents, and what they hold relative to
// the largest is the same).  A column where one is leaves a NaN as its first element, and the launch
// behind this one (attn_latent_block_kernel, which otherwise ends at once) takes its place.
constexpr int kLatColumns = 128;      // of a workgroup
constexpr float kLatRange = 60.f;

__device__ __forceinline__ unsigned lds_address(const void* p) {
  return (unsigned)(size_t)(__attribute__((address_space(3))) const void*)p;
}
// 16 bytes a lane from base + offset (base, lds the same in every lane) to lds + 16 * lane.
__device__ __forceinline__ void load_to_lds(unsigned lds, const void* base, unsigned offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
// The same from an address of the lane's own.
__device__ __forceinline__ void load_to_lds(unsigned lds, const void* address) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(address) : "memory", "m0");
}

template <int NB, int KS>   // latents of 32 NB elements, rows of 16 KS
__global__ __launch_bounds__(64 * kLatWaves) __attribute__((amdgpu_waves_per_eu(NB <= 4 ? 2 : 1))) void attn_latent_columns_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
    const int* __restrict__ positions, const int* __restrict__ span_of_token, const int* __restrict__ block_table,
    int max_pages, int page_size, unsigned page_magic, int n, int H, float scale, int window) {
  constexpr int rank = 32 * NB, row = 16 * KS, row8 = row / 8;
  constexpr int row_mask = row8 % 8 == 0 ? 7 : row8 % 4 == 0 ? 3 : 1;
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_tiles[];   // two buffers: [32][row], [rank][32]
  auto page_index = [&](int key) { return (int)(__umulhi((unsigned)key, page_magic) >> 3); };
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane / 32, c = lane % 32;
  constexpr int buf_elems = 32 * row + 32 * rank;
  // later tokens of a prompt read more keys: the workgroups with the most to do start first
  const long col0 = (long)(gridDim.x - 1 - blockIdx.x) * kLatColumns;
  const long ncols = (long)n * H;
  const int t_first = (int)(col0 / H), t_last = (int)((min(col0 + kLatColumns, ncols) - 1) / H);
  const long col = min(col0 + 32 * wave + c, ncols - 1);
  const bool col_ok = col0 + 32 * wave + c < ncols;
  const int t = (int)(col / H);
  const int my_span = span_of_token[t];
  const int len = positions[t] + 1;
  const int lo = first_key(len - 1, window, 0);
  const long page_elems = (long)page_size * (row + rank);
  const float c2 = scale * 1.4426950408889634f;             // scale * log2(e)
  bf16x8 qreg[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) qreg[kk] = *reinterpret_cast<const bf16x8*>(q + col * row + 16 * kk + 8 * g);

  float m = -INFINITY, l = 0.f;
  floatx16 acc[NB];
#pragma unroll
  for (int r = 0; r < NB; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.f;

  // ---- where this lane's pieces of a tile come from.  Rows: load j of the wave (every fourth one) fills the
  // 64 pieces from 64 (4 j + wave) on; a half (16 keys, 2 row8 whole loads) lies in one page.  Latents:
  // load j fills 16 elements' pieces; the lane's piece, and with it its half, is the same in all of them.
  constexpr int KL = KS / 4 + (KS % 4 ? 1 : 0);              // loads of a wave: 32 rows of 2 KS pieces over 256 lanes
  unsigned k_off[KL];
#pragma unroll
  for (int j = 0; j < KL; ++j) {
    const int piece = 64 * (4 * j + wave) + lane;
    const int kr = piece / row8, kp = piece - kr * row8;
    k_off[j] = (unsigned)(((kr % 16) * row + 8 * (kp ^ (kr & row_mask))) * (int)sizeof(bf16_t));
  }
  const int v_piece = (lane % 4) ^ (lane / 16 % 4), v_half = v_piece / 2;
  const int v_off = 8 * (v_piece % 2) + (16 * wave + lane / 4) * page_size;
  const unsigned lds0 = lds_address(lat_tiles);
  // ... and where it reads them: four places each, the rest are constant distances
  const int krow = (c & 19) | ((c & 4) << 1) | ((c & 8) >> 1);
  int k_at[4], v_at[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) k_at[j] = krow * row + 8 * ((2 * j + g) ^ (krow & row_mask));
#pragma unroll
  for (int u = 0; u < 2; ++u) v_at[u] = c * 32 + 8 * ((2 * u + g) ^ (c / 4 % 4));

  bool over = false;
  for (int first = t_first; first <= t_last;) {
    const int span = span_of_token[first];
    int last = first;
    while (last < t_last && span_of_token[last + 1] == span) ++last;
    const int group_len = positions[last] + 1;                // the span's last token here reads the most keys
    const int group_lo = first_key(positions[first], window, 0);   // ... and its first the earliest (pages before it may be gone)
    const bool mine = col_ok && my_span == span;
    const int* table = block_table + (long)span * max_pages;
    auto half_live = [&](int k0) { return k0 < group_len && k0 + 16 > group_lo; };
    struct Halves {
      int page[2];
    };
    // a vector load although the address is the same in every lane (see fetch: it has the loop's turn to arrive)
    auto lookup = [&](int kb) -> Halves {
      Halves P;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int index = half_live(kb + 16 * u) ? page_index(kb + 16 * u) : 0;
        asm volatile("" : "+v"(index));
        P.page[u] = table[index];
      }
      return P;
    };
    struct Source {
      const bf16_t *k[2], *v;                                 // the halves' rows; this lane's latents
      unsigned lds;
    };
    auto source = [&](int kb, const Halves& P, int buf) -> Source {
      const bf16_t* base[2];
      int slot[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k0 = kb + 16 * u;
        const bool live = half_live(k0);                      // a half that nobody reads takes page 0
        const int page = __builtin_amdgcn_readfirstlane(P.page[u]);
        base[u] = cache + (long)(live ? page : 0) * page_elems;
        slot[u] = live ? k0 - page_index(k0) * page_size : 0;
      }
      const bf16_t* v0 = base[0] + (long)page_size * row + slot[0];
      const bf16_t* v1 = base[1] + (long)page_size * row + slot[1];
      return {{base[0] + (long)slot[0] * row, base[1] + (long)slot[1] * row},
              (v_half ? v1 : v0) + v_off,
              lds0 + (unsigned)(buf * buf_elems) * (unsigned)sizeof(bf16_t)};
    };
    constexpr int LOADS = KL + NB / 2;                        // of a wave for a tile: rows, then latents
    auto fetch = [&](Source& F, int j) __attribute__((always_inline)) {
      if (j < KL) {
        const int load = 4 * j + wave;                        // of KS; the first KS / 2 are the first half's
        if (KS % 4 == 0 || load < KS) load_to_lds(F.lds + 1024u * (unsigned)load, F.k[2 * load >= KS], k_off[j < KL ? j : 0]);
      } else {
        const int load = 4 * (j - KL) + wave;                 // of 2 NB
        load_to_lds(F.lds + (unsigned)(32 * row) * (unsigned)sizeof(bf16_t) + 1024u * (unsigned)load, F.v);
        F.v += 64 * (long)page_size;
        asm volatile("" : "+v"(F.v));                         // (one address, not one for every load)
      }
    };
    const int kb0 = group_lo / 32 * 32;
    Halves pages = lookup(kb0);
    __syncthreads();                                          // the span before this one has been worked through
    {
      Source F = source(kb0, pages, 0);
#pragma unroll
      for (int j = 0; j < LOADS; ++j) fetch(F, j);
    }
    pages = lookup(kb0 + 32);
    int buf = 0;
    for (int kb = kb0; kb < group_len; kb += 32, buf ^= 1) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // this wave's part of the tile is in LDS, its reads of the last one are done
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      Source F = source(kb + 32, pages, buf ^ 1);       // (behind the last tile: halves that nobody reads)
      pages = lookup(kb + 64);
      bf16_t* const ks = lat_tiles + buf * buf_elems;         // [32][row]
      bf16_t* const vs = ks + 32 * row;                       // [rank][32]
      if (kb + 32 > group_len || !half_live(kb)) {            // latents of slots that may hold anything become zeros
        for (int i = tid; i < 32 * rank; i += 64 * kLatWaves) {
          const int key = kb + i % 32;
          if (key >= group_len || !half_live(kb + i % 32 / 16 * 16)) {
            const int e = i / 32, piece = i % 32 / 8;
            vs[e * 32 + 8 * (piece ^ (e / 4 % 4)) + i % 8] = (bf16_t)0.f;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      // ---- scores: this lane's key row is krow; the next tile's loads between the products (all at once in front of them they kept
      // the wave from its LDS reads)
      // (kAhead groups of pieces are on their way from LDS while one is multiplied, and no more: registers; two took 156 us where one takes 136)
      constexpr int kGroup = 2, kAhead = 1;
      floatx16 s0 = {}, s1 = {};
      bf16x8 ka[kAhead + 1][kGroup];
      auto read_k = [&](int kk) __attribute__((always_inline)) {           // piece 2 kk + g of the row, at its swapped place
        ka[kk / kGroup % (kAhead + 1)][kk % kGroup] = *reinterpret_cast<const bf16x8*>(ks + k_at[kk % 4] + 64 * (kk / 4));
      };
#pragma unroll
      for (int kk = 0; kk < kGroup * kAhead; ++kk)
        if (kk < KS) read_k(kk);
#pragma unroll
      for (int k0 = 0; k0 < KS; k0 += kGroup) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j)
          if (k0 + kGroup * kAhead + j < KS) read_k(k0 + kGroup * kAhead + j);
        __builtin_amdgcn_sched_barrier(0);
        s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[k0 / kGroup % (kAhead + 1)][0], qreg[k0], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[k0 / kGroup % (kAhead + 1)][1], qreg[k0 + 1], s1, 0, 0, 0);
        if (k0 / kGroup < LOADS) fetch(F, k0 / kGroup);
        __builtin_amdgcn_sched_barrier(0);
      }
      static_assert(LOADS <= KS / kGroup, "every load has its group");
      bf16x8 va[kAhead + 1][2];
      auto read_v = [&](int r) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) va[r % (kAhead + 1)][u] = *reinterpret_cast<const bf16x8*>(vs + v_at[u] + 1024 * r);
      };
#pragma unroll
      for (int r = 0; r < kAhead; ++r)
        if (r < NB) read_v(r);
      const int hi_e = mine ? len - 1 - kb - 8 * g : -1, lo_e = lo - kb - 8 * g;    // offsets that this lane's column reads
      float tmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int e = 16 * (i / 8) + i % 8;
        s0[i] = (e <= hi_e && e >= lo_e) ? (s0[i] + s1[i]) * c2 : -INFINITY;
        tmax = fmaxf(tmax, s0[i]);
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
      if (m == -INFINITY) m = tmax;                           // the column's first keys
      over |= tmax > m + kLatRange;
      const float mref = m == -INFINITY ? 0.f : m;            // (a column without a key so far: every score is -inf)
      bf16x8 pb[2];
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bf16_t p = (bf16_t)__builtin_amdgcn_exp2f(s0[i] - mref);      // exp2(-inf) = 0
        pb[i / 8][i % 8] = p;
        psum += (float)p;
      }
      l += psum;
      // ---- the weighted sum of the latents
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        if (r + kAhead < NB) read_v(r + kAhead);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[r % (kAhead + 1)][u], pb[u], acc[r], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // nothing more comes into LDS (the last tile's loads went to the other buffer)
    first = last + 1;
  }
  l += __shfl_xor(l, 32, kWave);
  if (!col_ok) return;
  const float inv = over ? NAN : 1.f / l;
  bf16_t* orow = out + col * rank;
  float none = 0.f;                                           // 0, or NaN where an element is not finite
#pragma unroll
  for (int r = 0; r < NB; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float o = acc[r][4 * b + i] * inv;
        v[i] = (bf16_t)o;
        none = fmaf(o, 0.f, none);
      }
      *reinterpret_cast<bf16x4*>(orow + 32 * r + 8 * b + 4 * g) = v;
    }
  // Where the columns are several requests', all of them were multiplied by the latents of all, by probabilities of 0, which a NaN or an infinity comes
  // through: such a column goes to the launch behind, which keeps requests apart.  (Known only here, from the spans' list: a flag along the loop, or a
  // branch for waves without a column in a tile, sends registers of ranks of 512 through scratch memory, 1,500 tokens of 32 heads 137 -> 152 and 816 us.)
  none += __shfl_xor(none, 32, kWave);
  if (isnan(none) && span_of_token[t_first] != span_of_token[t_last] && g == 0) *orow = (bf16_t)NAN;
}

template <int NB, int KS>
static int launch_latent_columns(const void* q, void* out, const void* cache, const int* positions, const int* span_of_token,
                                 const int* block_table, int max_pages, int page_size, int n, int H, float scale, int window,
                                 hipStream_t stream) {
  const size_t lds = 2 * (size_t)(32 * 16 * KS + 32 * 32 * NB) * sizeof(bf16_t);
  static size_t raised_to = 64 * 1024;
  if (lds > raised_to) {
    hipError_t e = hipFuncSetAttribute((const void*)attn_latent_columns_kernel<NB, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) KLLM_FAIL((int)e, "attn_latent: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised_to = lds;
  }
  const unsigned page_magic = (unsigned)(((1ull << 35) + page_size - 1) / page_size);
  hipLaunchKernelGGL((attn_latent_columns_kernel<NB, KS>), dim3(ceil_div((long)n * H, kLatColumns)), dim3(64 * kLatWaves), lds, stream,
                     (const bf16_t*)q, (bf16_t*)out, (const bf16_t*)cache, positions, span_of_token, block_table, max_pages,
                     page_size, page_magic, n, H, scale, window);
  return 0;
}

// The slices' results of one (token, head) become its output: weights exp2(m_s - max m).  Lane s takes slice s's maximum and sum and works
// out its weight, each wave for itself; every slice's outputs are asked for behind them, so that all of it is one trip to memory (weights
// first and then eight slices at a time: 9.6 us for 8 tokens, 32 heads and 32 slices of 512; so 4.9 with 16).  R: at least the number of slices.
template <int R>
__global__ __launch_bounds__(kLatThreads) void attn_latent_merge_kernel(const float* __restrict__ part, int rank, int nslices,
                                                                        bf16_t* __restrict__ out) {
  const int lane = threadIdx.x % kWave, bytes = (rank + 2) * (int)sizeof(float);
  const long th = blockIdx.x;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(part)) + th * nslices * bytes, 0, nslices * bytes, 0x00020000);
  // (beyond the last slice zeros, from nowhere: all of a place is in the vector offset, which the descriptor's end is held against)
  auto load = [&](int at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rows, at, 0, 0)); };
  const float m0 = load(lane * bytes + 4 * rank), ls = load(lane * bytes + 4 * rank + 4);
  float v[2][R];
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) v[e][j] = load(4 * min((int)threadIdx.x + e * kLatThreads, rank - 1) + j * bytes);
  __builtin_amdgcn_sched_barrier(0);
  const float ms = lane < nslices ? m0 : -INFINITY;
  const float M = first_lanes_max<R>(ms);                     // finite: some slice holds the token's own key
  const float w = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - M);
  const float wn = w / wave_sum(w * ls);                      // 0 for a slice without a key, whose outputs may be anything
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) asm volatile("" : "+v"(v[e][j]));
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    float o = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float wj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wn), j));
      o = fmaf(wj, wj == 0.f ? 0.f : v[e][j], o);
    }
    const int at = threadIdx.x + e * kLatThreads;
    if (at < rank) out[th * rank + at] = (bf16_t)o;
  }
}

template <int NR, int KS>
static void launch_latent_mfma(const void* q, void* out, const void* cache, const int* positions, const int* span_of_token,
                               const int* block_table, int max_pages, int page_size, int n, int H, int row, int rank,
                               float scale, int window, float* part, int nslices, int redo, hipStream_t stream) {
  if (nslices == 0) {       // steps of many tokens: four tokens a workgroup, their keys through LDS
    const unsigned page_magic = (unsigned)(((1ull << 35) + page_size - 1) / page_size);
    const size_t tiles = ((size_t)32 * (row + 8) + (size_t)rank * 36) * sizeof(bf16_t);
    static size_t raised_to = 64 * 1024;
    if (tiles > raised_to) {
      (void)hipFuncSetAttribute((const void*)attn_latent_block_kernel<NR, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)tiles);
      raised_to = tiles;
    }
    hipLaunchKernelGGL((attn_latent_block_kernel<NR, KS>), dim3((n + kLatWaves - 1) / kLatWaves, (H + 15) / 16), dim3(64 * kLatWaves),
                       tiles, stream, (const bf16_t*)q, (bf16_t*)out, (const bf16_t*)cache, positions, span_of_token,
                       block_table, max_pages, page_size, page_magic, n, H, row, rank, scale, window, redo);
    return;
  }
  const unsigned page16 = page_size / 16, magic16 = page16 == 1 ? 0xFFFFFFFFu : (unsigned)((1ull << 32) / page16);
  hipLaunchKernelGGL((attn_latent_mfma_kernel<NR, KS>), dim3(n, (H + 15) / 16, nslices), dim3(64 * kLatWaves), 0, stream,
                     (const bf16_t*)cache, positions, span_of_token, block_table, (const bf16_t*)q, max_pages, (int)page16, H, row, rank,
                     magic16, scale, window, nslices, (bf16_t*)out, part);
#define KLLM_LATM(R) hipLaunchKernelGGL(attn_latent_merge_kernel<R>, dim3(n * H), dim3(kLatThreads), 0, stream, part, rank, nslices, (bf16_t*)out)
  if (nslices > 32) KLLM_LATM(64);
  else if (nslices > 16) KLLM_LATM(32);
  else if (nslices > 1) KLLM_LATM(16);
#undef KLLM_LATM
}

// attended: [n][H][rank]; w_uv [H * dv][rank]; gate: [nsplit][n][H * dv] sums ([H] with by_head) or null.
template <typename T>
__global__ __launch_bounds__(kLatThreads) void latent_out_kernel(
    const T* __restrict__ attended, const T* __restrict__ w_uv, const float* __restrict__ gate, int nsplit,
    long split_stride, long gate_stride, int by_head, T* __restrict__ out, int H, int dv, int rank) {
  extern __shared__ float al[];          // [rank]
  const long t = blockIdx.x;
  const int h = blockIdx.y, tid = threadIdx.x;
  const T* src = attended + (t * H + h) * rank;
  for (int i = tid; i < rank; i += kLatThreads) al[i] = to_f32(src[i]);
  __syncthreads();
  for (int j = tid; j < dv; j += kLatThreads) {
    const T* w = w_uv + ((long)h * dv + j) * rank;
    float acc = 0.f;
    for (int r = 0; r < rank; ++r) acc = fmaf(al[r], to_f32(w[r]), acc);
    const long col = (long)h * dv + j;
    if (gate) {
      float g = 0.f;
      for (int s = 0; s < nsplit; ++s) g += gate[s * split_stride + t * gate_stride + (by_head ? h : col)];
      acc *= sigmoid_f32(g);
    }
    out[t * H * dv + col] = from_f32<T>(acc);
  }
}

// The two products with a head's own matrix on the matrix cores (bfloat16), MFMA 16x16x32 as
// above: a wave takes 16 outputs (rows of the head's matrix, one per lane, 16 bytes at a time)
// and 16 tokens, latent_query's workgroups four such pieces of 16 outputs.
//   latent_out:   out[t][h][j] = sum_r W_uv[h dv + j][r] attended[t][h][r], times the gate
//   latent_query: out[t][h][r] = sum_i W_ukT[h][r][i] q[t][h][i] (W_ukT: the head's matrix
//                 transposed once, when the weights are bound), and the rotated part beside it
// What bounds a decode batch's: trips to memory in a row.  So a wave asks for all it needs at once (up to 512 of the rank, the gate's
// sums; 128 of a head's, the rotated part), with arguments that came with the launch, and latent_out's waves are workgroups of
// their own, over four times the CUs.  8 tokens, 32 heads of 128, rank 512 + 64: both 9.4 -> 4.2 us (step
// after step, and a loop over the slices for every sum, before).
__global__ __launch_bounds__(kWave) void latent_out_mfma_kernel(
    const bf16_t* __restrict__ attended, const bf16_t* __restrict__ w_uv, int n, int H, int dv, int rank, const float* __restrict__ gate, long gate_stride,
    int nsplit, int by_head, long split_stride, bf16_t* __restrict__ out) {
  const int lane = threadIdx.x, g = lane / 16, c = lane % 16;
  const int h = blockIdx.y, j0 = blockIdx.z * 16;
  const int tt = blockIdx.x * 16 + c, t = min(tt, n - 1);
  const bf16_t* wrow = w_uv + ((long)h * dv + min(j0 + c, dv - 1)) * rank + 8 * g;
  const bf16_t* arow = attended + ((long)t * H + h) * rank + 8 * g;
  constexpr int STEPS = 8;                                 // of 32, asked for at once
  bf16x8 a[2][STEPS], b[2][STEPS];
  auto ask = [&](int k0, bf16x8 (&A)[STEPS], bf16x8 (&B)[STEPS]) {       // rank % 32 == 0 (the launch); beyond it the first, not used
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int k = k0 + 32 * i < rank ? k0 + 32 * i : 0;
      A[i] = *reinterpret_cast<const bf16x8*>(wrow + k);
      B[i] = *reinterpret_cast<const bf16x8*>(arow + k);
    }
  };
  ask(0, a[0], b[0]);
  if (rank > 32 * STEPS) ask(32 * STEPS, a[1], b[1]);
  float gs[4] = {0.f, 0.f, 0.f, 0.f}, more[4] = {0.f, 0.f, 0.f, 0.f};      // two slices of the gate's sums
  if (gate)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* at = gate + t * gate_stride + (by_head ? h : (long)h * dv + min(j0 + 4 * g + i, dv - 1));
      gs[i] = at[0];
      if (nsplit > 1) more[i] = at[split_stride];
    }
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < rank; k0 += 64 * STEPS) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (k0 + half * 32 * STEPS >= rank) break;
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
        if (k0 + 32 * (half * STEPS + i) < rank) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[half][i], b[half][i], acc, 0, 0, 0);
      if (k0 + 32 * STEPS * (half + 2) < rank) ask(k0 + 32 * STEPS * (half + 2), a[half], b[half]);
    }
  }
  if (tt >= n) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int jj = j0 + 4 * g + i;
    if (jj >= dv) continue;
    const long col = (long)h * dv + jj;
    float v = acc[i];
    if (gate) {
      gs[i] += more[i];
      for (int s = 2; s < nsplit; ++s) gs[i] += gate[s * split_stride + tt * gate_stride + (by_head ? h : col)];
      v *= sigmoid_f32(gs[i]);
    }
    out[(long)tt * H * dv + col] = (bf16_t)v;
  }
}

__global__ __launch_bounds__(kLatThreads) void latent_query_mfma_kernel(
    const float* __restrict__ q, const bf16_t* __restrict__ w_ukt, int n, int H, int d, int dr, int rank, int nsplit,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, bf16_t* __restrict__ out, long split_stride) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int g = lane / 16, c = lane % 16;
  const int h = blockIdx.y;
  const int hw = d + dr, half = dr / 2;
  const int t = min((int)blockIdx.x * 16 + c, n - 1);
  const int tt = blockIdx.x * 16 + c;
  const float* in = q + ((long)t * H + h) * hw;
  const int r0 = (blockIdx.z * 4 + wave) * 16;
  // Everything that a wave needs is asked for before anything is used, 128 of d at a time: weights, the heads' sums, and its
  // share of the rotated part (elements 4 piece + g and every 16 gridDim.z'th behind).
  typedef float anywhere4 __attribute__((ext_vector_type(4), aligned(4)));      // (rows of d + dr floats)
  const bf16_t* wrow = w_ukt + ((long)h * rank + min(r0 + c, rank - 1)) * d;
  constexpr int STEPS = 4;
  bf16x8 w[STEPS];
  floatx4 x[STEPS][2];
  auto ask = [&](int k0) {
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      if (i == 2 && k0 + 64 >= d) break;                     // (d a multiple of 32; beyond it the step's own first, not used)
      const int k = (k0 + 32 * i < d ? k0 + 32 * i : k0) + 8 * g;
      w[i] = *reinterpret_cast<const bf16x8*>(wrow + k);
#pragma unroll
      for (int j = 0; j < 2; ++j) x[i][j] = *reinterpret_cast<const anywhere4*>(in + k + 4 * j);
    }
  };
  if (r0 < rank) ask(0);
  bf16_t* dst = out + ((long)tt * H + h) * (rank + dr);
  for (int i = (blockIdx.z * 4 + wave) * 4 + g; i < half; i += 16 * gridDim.z) {
    float u = in[d + i], v = in[d + half + i];
    const float cs = cos_t[(long)t * half + i], sn = sin_t[(long)t * half + i];
    for (int s = 1; s < nsplit; ++s) {
      u += in[s * split_stride + d + i];
      v += in[s * split_stride + d + half + i];
    }
    if (tt < n) {
      dst[rank + i] = (bf16_t)(u * cs - v * sn);
      dst[rank + half + i] = (bf16_t)(v * cs + u * sn);
    }
  }
  if (r0 >= rank) return;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < d; k0 += 32 * STEPS) {
    if (k0) ask(k0);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      if (k0 + 32 * i >= d) break;
      for (int s = 1; s < nsplit; ++s)
#pragma unroll
        for (int j = 0; j < 2; ++j) x[i][j] += *reinterpret_cast<const anywhere4*>(in + s * split_stride + k0 + 32 * i + 8 * g + 4 * j);
      bf16x8 b;
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = (bf16_t)x[i][e / 4][e % 4];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], b, acc, 0, 0, 0);
    }
  }
  if (tt >= n) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (r0 + 4 * g + i < rank) dst[r0 + 4 * g + i] = (bf16_t)acc[i];
}

// The same two products for steps of many tokens, MFMA 32x32x16 (lane l: g = l/32, c = l%32: A[c][8g..],
// B[8g..][c], D[8(i/4) + 4g + i%4][c]): a workgroup takes 64 tokens of a head, A = 32 outputs (rows of the
// head's matrix), B = 32 tokens; a lane then holds pieces of four neighbouring outputs of one token.
constexpr int kLatTokens = 64;

// DS = d / 16.  The tokens' queries (their slices added, in the compute type) pass through LDS once
// for all outputs; a wave takes every fourth piece of 32 outputs.
template <int DS>
__global__ __launch_bounds__(kLatThreads, DS <= 8 ? 4 : 2) void latent_query_block_kernel(
    const float* __restrict__ q, int nsplit, long split_stride, const bf16_t* __restrict__ w_ukt,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, bf16_t* __restrict__ out, int n, int H, int dr,
    int rank) {
  constexpr int d = 16 * DS, LD = d + 8;
  __shared__ __attribute__((aligned(16))) bf16_t qs[kLatTokens * LD];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int g = lane / 32, c = lane % 32;
  const int h = blockIdx.x, t0 = blockIdx.y * kLatTokens;
  const int hw = d + dr, half = dr / 2;
  const long row_out = (long)H * (rank + dr);
  // A thread asks for a slice of its pieces together, up to eight at a time (one after the other, a trip to memory each: a prompt
  // of 70 tokens at Natenex sizes 995 us, now 961, of 200 1,256 / 1,240; of 1,500, where other workgroups fill the wait, 34.9 / 33.5 of a layer).
  typedef float anywhere4 __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int PIECES = kLatTokens * (d / 4), MANY = DS < 8 ? DS : 8;        // (DS pieces a thread)
#pragma unroll 1
  for (int i0 = tid; i0 < PIECES; i0 += MANY * kLatThreads) {
    floatx4 v[MANY];
    for (int s = 0; s < nsplit; ++s) {
      floatx4 x[MANY];
#pragma unroll
      for (int k = 0; k < MANY; ++k) {
        const int i = min(i0 + k * kLatThreads, PIECES - 1), tt = i / (d / 4), e = 4 * (i % (d / 4));
        x[k] = *reinterpret_cast<const anywhere4*>(q + s * split_stride + ((long)min(t0 + tt, n - 1) * H + h) * hw + e);
      }
#pragma unroll
      for (int k = 0; k < MANY; ++k) v[k] = s == 0 ? x[k] : v[k] + x[k];
    }
#pragma unroll
    for (int k = 0; k < MANY; ++k) {
      const int i = i0 + k * kLatThreads, tt = i / (d / 4), e = 4 * (i % (d / 4));
      if (i < PIECES) *reinterpret_cast<bf16x4*>(qs + tt * LD + e) = bf16x4{(bf16_t)v[k][0], (bf16_t)v[k][1], (bf16_t)v[k][2], (bf16_t)v[k][3]};
    }
  }
  // the rotated part beside it, as many pairs a thread at a time as there are
  const int pairs = kLatTokens * half;
  auto rotated = [&](auto at_a_time) {
    constexpr int PAIRS = decltype(at_a_time)::value;
#pragma unroll 1
    for (int i0 = tid; i0 < pairs; i0 += PAIRS * kLatThreads) {
      float u[PAIRS], v[PAIRS], cs[PAIRS], sn[PAIRS];
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) {
        const int i = min(i0 + k * kLatThreads, pairs - 1), tt = i / half, e = i - tt * half, t = min(t0 + tt, n - 1);
        const float* in = q + ((long)t * H + h) * hw + d + e;
        u[k] = in[0];
        v[k] = in[half];
        cs[k] = cos_t[(long)t * half + e];
        sn[k] = sin_t[(long)t * half + e];
      }
      for (int s = 1; s < nsplit; ++s)
#pragma unroll
        for (int k = 0; k < PAIRS; ++k) {
          const int i = min(i0 + k * kLatThreads, pairs - 1), tt = i / half, e = i - tt * half, t = min(t0 + tt, n - 1);
          const float* in = q + s * split_stride + ((long)t * H + h) * hw + d + e;
          u[k] += in[0];
          v[k] += in[half];
        }
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) {
        const int i = i0 + k * kLatThreads, tt = i / half, e = i - tt * half, t = t0 + tt;
        if (i >= pairs || t >= n) continue;
        bf16_t* dst = out + t * row_out + (long)h * (rank + dr) + rank + e;
        dst[0] = (bf16_t)(u[k] * cs[k] - v[k] * sn[k]);
        dst[half] = (bf16_t)(v[k] * cs[k] + u[k] * sn[k]);
      }
    }
  };
  if (half <= 8) rotated(std::integral_constant<int, 2>()); else rotated(std::integral_constant<int, 8>());
  __syncthreads();
  for (int r0 = 32 * wave; r0 < rank; r0 += 32 * (kLatThreads / kWave)) {
    const bf16_t* wrow = w_ukt + ((long)h * rank + min(r0 + c, rank - 1)) * d + 8 * g;
    bf16x8 a[DS];
#pragma unroll
    for (int k = 0; k < DS; ++k) a[k] = *reinterpret_cast<const bf16x8*>(wrow + 16 * k);
#pragma unroll
    for (int tb = 0; tb < kLatTokens / 32; ++tb) {
      floatx16 acc = {};
#pragma unroll
      for (int k = 0; k < DS; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[k], *reinterpret_cast<const bf16x8*>(qs + (32 * tb + c) * LD + 16 * k + 8 * g),
                                                      acc, 0, 0, 0);
      const int t = t0 + 32 * tb + c;
      if (t >= n) continue;
      bf16_t* dst = out + t * row_out + (long)h * (rank + dr) + r0 + 4 * g;
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (r0 + 8 * b + 4 * g < rank)                        // rank in steps of 4 (the launch)
          *reinterpret_cast<bf16x4*>(dst + 8 * b) =
              bf16x4{(bf16_t)acc[4 * b], (bf16_t)acc[4 * b + 1], (bf16_t)acc[4 * b + 2], (bf16_t)acc[4 * b + 3]};
    }
  }
}

// A workgroup takes 64 tokens of a head and 64 U of its outputs, a wave 16 U of those (U 2, or 1 where that leaves CUs without work).  The tokens' rows of up to 512 of the rank go into LDS, a row a load
// instruction (they lie H rank apart: a matrix operand's lanes would ask for 32 bytes of 32 rows, 32 pages, a load; the tiles of all
// products, which come back to a row for every 128 bytes, took 8 to 20 us more than that up to 200 tokens),
// and a wave's weights into registers, all on their way at once.  Chunk j (16 bytes) of row r lies in slot j ^ (r % 16), so that sixteen rows' chunk
// meets all banks.  Row c of the u-th of a wave's A operands is output 4 U (c / 4) + 4 u + c % 4: a lane then holds 4 U neighbouring
// outputs of a token.  In us, 32 heads of 128, rank 512, with a gate in one slice, operands by lane before and now: 64 tokens 11.8 -> 9.1, 200 12.2 ->
// 9.4, 260 21.0 -> 12.3, 400 21.5 -> 12.7, 700 31.1 -> 20.8, 1,500 60.4 -> 33.4, in four slices 17.1 -> 11.5, 17.9 -> 13.7, 31.0 -> 17.5, 31.8 -> 19.3, 48.1 ->
// 29.9, 96.7 -> 47.7; U 2 / 1: 200 tokens 13.1 / 9.4, 400 13.6 / 12.7, 520 (288 workgroups of U 2) 16.1 / 19.8, 1,500 33.4 / 40.3.
// CHUNK: of the rank, in LDS and registers at a time.  With 512 whatever the rank, rows of 64 to 256 asked for what they do not have: us, operands by lane, 512, and
// so: rank 64 (4 heads of 64, 200 tokens) 4.4, 6.1, 3.6; 96 (33 of 40, 1,500) 7.4, 12.6, 5.2; 256 (16 of 128, 500) 6.5, 7.2, 5.3.  Heads of up to 64 outputs take U 1.
template <int U, int CHUNK>
__global__ __launch_bounds__(kLatThreads, 2) void latent_out_block_kernel(
    const bf16_t* __restrict__ attended, const bf16_t* __restrict__ w_uv, int n, int H, int dv, int rank, const float* __restrict__ gate, long gate_stride,
    int nsplit, int by_head, long split_stride, bf16_t* __restrict__ out) {
  constexpr int STEPS = CHUNK / 32, TB = kLatTokens / 16, SLOTS = CHUNK / 8;
  __shared__ __attribute__((aligned(1024))) bf16_t rows[kLatTokens * CHUNK];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 16, c = lane % 16;
  const int h = blockIdx.x, t0 = blockIdx.y * kLatTokens, j0 = 16 * U * (4 * blockIdx.z + wave);
  const bf16_t* wrow[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wrow[u] = w_uv + ((long)h * dv + min(j0 + 4 * U * (c / 4) + 4 * u + c % 4, dv - 1)) * rank;
  floatx4 acc[TB][U];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb)
#pragma unroll
    for (int u = 0; u < U; ++u) acc[tb][u] = floatx4{0.f, 0.f, 0.f, 0.f};
  typedef float anywhere4 __attribute__((ext_vector_type(4), aligned(4)));
  auto opened = [&](int s, floatx4 (&z)[TB][U]) {           // a slice of the gate's sums for this lane's outputs
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const float* at = gate + s * split_stride + min(t0 + 16 * tb + c, n - 1) * gate_stride;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (by_head) {
          const float one = at[h];
          z[tb][u] = floatx4{one, one, one, one};
        } else {                                              // (pieces behind the head's outputs: its last one, not used)
          const int j = j0 + 4 * U * g + 4 * u;
          if (dv % 4 == 0) {
            z[tb][u] = *reinterpret_cast<const anywhere4*>(at + (long)h * dv + min(j, dv - 4));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) z[tb][u][e] = at[(long)h * dv + min(j + e, dv - 1)];
          }
        }
      }
    }
  };
  floatx4 z[TB][U];
  for (int k0 = 0; k0 < rank; k0 += CHUNK) {
    const int width = min(rank - k0, CHUNK), chunks = width / 8;       // rank % 16 == 0 (the launch)
    if (k0) __syncthreads();
#pragma unroll
    for (int i = 0; i < kLatTokens / 4 / (kWave / SLOTS); ++i) {
      const int r0 = (4 * i + wave) * (kWave / SLOTS), r = r0 + lane / SLOTS;
      const int chunk = lane % SLOTS ^ (r % 16);                          // (chunks that are not there are never read)
      const bf16_t* src = attended + ((long)min(t0 + r, n - 1) * H + h) * rank + k0 + 8 * (chunk < chunks ? chunk : 0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(rows + r0 * CHUNK), 16, 0, 0);
    }
    bf16x8 w[U][STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int u = 0; u < U; ++u) w[u][s] = *reinterpret_cast<const bf16x8*>(wrow[u] + k0 + (32 * s + 8 * g < width ? 32 * s + 8 * g : 0));
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int u = 0; u < U; ++u) asm volatile("" : "+v"(w[u][s]));       // (here, not step by step behind the barrier)
    if (U == 1 && gate && k0 == 0) opened(0, z);           // (two operands' weights leave no registers for it)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's rows are in LDS: a barrier alone waits for no load from memory
    __syncthreads();
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      if (32 * s >= width) break;
      const bool there = 32 * s + 8 * g < width;             // (half a step where the rank is no multiple of 32: zeros)
      const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const int r = 16 * tb + c;
        bf16x8 b = *reinterpret_cast<const bf16x8*>(rows + r * CHUNK + 8 * ((4 * s + g) ^ c));
        b = there ? b : zero;
#pragma unroll
        for (int u = 0; u < U; ++u) acc[tb][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(there ? w[u][s] : zero, b, acc[tb][u], 0, 0, 0);
      }
    }
  }
  constexpr int E = 4 * U;
  if (j0 + E * g >= dv) return;
  typedef bf16_t piece __attribute__((ext_vector_type(E)));
  const bool whole = dv % E == 0 && ((unsigned long)out & (2 * E - 1)) == 0;
  if (U > 1 && gate) opened(0, z);
  for (int s = 1; gate && s < nsplit; ++s) {                  // (a slice's sums all together)
    floatx4 more[TB][U];
    opened(s, more);
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int u = 0; u < U; ++u) z[tb][u] += more[tb][u];
  }
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    const int t = t0 + 16 * tb + c;
    if (t >= n) continue;
    piece v;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      float a = acc[tb][e / 4][e % 4];
      if (gate) a *= sigmoid_f32(z[tb][e / 4][e % 4]);
      v[e] = (bf16_t)a;
    }
    bf16_t* dst = out + ((long)t * H + h) * dv + j0 + E * g;
    if (whole) {
      *reinterpret_cast<piece*>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (j0 + E * g + e < dv) dst[e] = v[e];
    }
  }
}

}  // namespace kllm

using namespace kllm;

extern "C" int kllm_latent_max_row(void) { return kLatMaxRow; }

extern "C" int kllm_latent_kv_append(const float* dkv, int nsplit, long split_stride, const float* weight, float eps,
                                     const float* cos_t, const float* sin_t, void* cache, const int* positions,
                                     const int* span_of_token, const int* block_table, int max_pages, int page_size,
                                     int n, int rank, int dr, int dtype, long in_stride, hipStream_t stream) {
  KLLM_REQUIRE(dkv && weight && cos_t && sin_t && cache && positions && span_of_token && block_table,
               "latent_kv_append: null pointer");
  KLLM_REQUIRE(n > 0 && nsplit >= 1 && rank > 0 && dr > 0 && dr % 2 == 0 && rank + dr <= kLatMaxRow,
               "latent_kv_append: bad sizes n=%d rank=%d dr=%d (rows of up to %d)", n, rank, dr, kLatMaxRow);
  KLLM_REQUIRE(max_pages > 0 && page_size > 0, "latent_kv_append: bad cache sizes");
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "latent_kv_append: unknown dtype %d", dtype);
#define KLLM_LK(T, PER)                                                                                                  \
  hipLaunchKernelGGL((latent_kv_append_kernel<T, PER>), dim3(n), dim3(kLatThreads), 0, stream, positions, span_of_token, \
                     dkv, in_stride, rank, dr, weight, block_table, max_pages, page_size, cos_t, sin_t, nsplit,          \
                     split_stride, eps, (T*)cache)
#define KLLM_LKS(T)                                                            \
  do {                                                                         \
    if (rank <= 2 * kLatThreads) KLLM_LK(T, 2); else KLLM_LK(T, kLatMaxPer);   \
  } while (0)
  if (dtype == DT_F32) KLLM_LKS(float); else KLLM_LKS(bf16_t);
#undef KLLM_LKS
#undef KLLM_LK
  KLLM_CHECK_LAUNCH("latent_kv_append");
  return 0;
}

extern "C" int kllm_latent_norm(const float* in, int nsplit, long split_stride, long in_stride, const float* weight,
                                float eps, void* out, int n, int r, int dtype, hipStream_t stream) {
  KLLM_REQUIRE(in && weight && out && n > 0 && r > 0 && nsplit >= 1 && in_stride >= r, "latent_norm: null pointer or bad sizes");
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "latent_norm: unknown dtype %d", dtype);
#define KLLM_LN(T, PER)                                                                                              \
  hipLaunchKernelGGL((latent_norm_kernel<T, PER>), dim3(n), dim3(kLatThreads), 0, stream, in, weight, in_stride, r,  \
                     nsplit, (T*)out, eps, split_stride)
#define KLLM_LNS(T)                                                        \
  do {                                                                     \
    if (r <= 4 * kLatThreads) KLLM_LN(T, 4);                               \
    else if (r <= 8 * kLatThreads) KLLM_LN(T, 8);                          \
    else if (r <= 16 * kLatThreads) KLLM_LN(T, 16);                        \
    else KLLM_LN(T, 0);                                                    \
  } while (0)
  if (dtype == DT_F32) KLLM_LNS(float); else KLLM_LNS(bf16_t);
#undef KLLM_LNS
#undef KLLM_LN
  KLLM_CHECK_LAUNCH("latent_norm");
  return 0;
}

extern "C" int kllm_latent_query(const float* q, int nsplit, long split_stride, const void* w_uk, const float* cos_t,
                                 const float* sin_t, void* out, int n, int H, int d, int dr, int rank, int dtype,
                                 int transposed, hipStream_t stream) {
  KLLM_REQUIRE(q && w_uk && cos_t && sin_t && out, "latent_query: null pointer");
  KLLM_REQUIRE(n > 0 && nsplit >= 1 && H > 0 && H <= 65535 && d > 0 && dr > 0 && dr % 2 == 0 && rank > 0 &&
                   rank + dr <= kLatMaxRow && d + dr <= 4096,
               "latent_query: bad sizes n=%d H=%d d=%d dr=%d rank=%d", n, H, d, dr, rank);
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "latent_query: unknown dtype %d", dtype);
  if (transposed) {     // w_uk is [H][rank][d]: the kernel on the matrix cores
    KLLM_REQUIRE(dtype == DT_BF16 && d % 32 == 0 && ((uintptr_t)w_uk & 15) == 0,
                 "latent_query: the transposed matrix goes with bfloat16 and head sizes in steps of 32 (d=%d)", d);
    if (n >= kLatTokens && rank % 4 == 0 && dr % 4 == 0 && d <= 256 && ((uintptr_t)out & 7) == 0 && (n + kLatTokens - 1) / kLatTokens <= 65535) {
      const dim3 grid(H, (n + kLatTokens - 1) / kLatTokens);
#define KLLM_LQ(DS)                                                                                                   \
  case DS / 2:                                                                                                        \
    hipLaunchKernelGGL(latent_query_block_kernel<DS>, grid, dim3(kLatThreads), 0, stream, q, nsplit, split_stride,    \
                       (const bf16_t*)w_uk, cos_t, sin_t, (bf16_t*)out, n, H, dr, rank);                              \
    break
      switch (d / 32) { KLLM_LQ(2); KLLM_LQ(4); KLLM_LQ(6); KLLM_LQ(8); KLLM_LQ(10); KLLM_LQ(12); KLLM_LQ(14); KLLM_LQ(16); }
#undef KLLM_LQ
      KLLM_CHECK_LAUNCH("latent_query");
      return 0;
    }
    hipLaunchKernelGGL(latent_query_mfma_kernel, dim3((n + 15) / 16, H, (rank + 63) / 64), dim3(kLatThreads), 0, stream, q,
                       (const bf16_t*)w_uk, n, H, d, dr, rank, nsplit, cos_t, sin_t, (bf16_t*)out, split_stride);
    KLLM_CHECK_LAUNCH("latent_query");
    return 0;
  }
  const size_t lds = (size_t)(d + dr) * sizeof(float);
  if (dtype == DT_F32)
    hipLaunchKernelGGL(latent_query_kernel<float>, dim3(n, H), dim3(kLatThreads), lds, stream, q, nsplit, split_stride,
                       (const float*)w_uk, cos_t, sin_t, (float*)out, H, d, dr, rank);
  else
    hipLaunchKernelGGL(latent_query_kernel<bf16_t>, dim3(n, H), dim3(kLatThreads), lds, stream, q, nsplit, split_stride,
                       (const bf16_t*)w_uk, cos_t, sin_t, (bf16_t*)out, H, d, dr, rank);
  KLLM_CHECK_LAUNCH("latent_query");
  return 0;
}

extern "C" int kllm_attn_latent(const void* q, void* out, const void* cache, const int* positions,
                                const int* span_of_token, const int* block_table, int max_pages, int page_size, int n,
                                int H, int row, int rank, float scale, int dtype, int mode, float* part, long part_floats, int nslices,
                                int window, hipStream_t stream) {
  KLLM_REQUIRE(q && out && cache && positions && span_of_token && block_table, "attn_latent: null pointer");
  KLLM_REQUIRE(n > 0 && H > 0 && H <= 65535 && rank > 0 && rank <= row && row <= kLatMaxRow,
               "attn_latent: bad sizes n=%d H=%d row=%d rank=%d (rows of up to %d)", n, H, row, rank, kLatMaxRow);
  KLLM_REQUIRE(max_pages > 0 && page_size > 0 && window >= 0, "attn_latent: bad cache sizes or window");
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "attn_latent: unknown dtype %d", dtype);
  if (dtype == DT_BF16 && mode != 1 && rank % 16 == 0 && row % 8 == 0 && rank <= 512 && page_size % 16 == 0 &&
      page_size <= 2048 && (long)max_pages * page_size <= (1L << 24) &&
      ((uintptr_t)q & 15) == 0 && ((uintptr_t)cache & 15) == 0 && ((uintptr_t)out & 7) == 0) {
    KLLM_REQUIRE(nslices >= 0 && nslices <= 64 && (nslices <= 1 || (part && ((uintptr_t)part & 7) == 0 && part_floats >= (long)n * H * nslices * (rank + 2))),
                 "attn_latent: %d slices need room for %d tokens x %d heads x %d slices x (%d + 2) floats", nslices, n, H,
                 nslices, rank);
    int redo = 0;
    if (nslices == 0 && (long)n * H / kLatColumns < (1L << 30)) {
      // the sizes that are built for long steps: (rank, row) = 32 NB, 16 KS
#define KLLM_LATC(NB, KS)                                                                                               \
  if (rank == 32 * NB && row == 16 * KS) {                                                                              \
    if (int rc = launch_latent_columns<NB, KS>(q, out, cache, positions, span_of_token, block_table, max_pages, page_size, n, \
                                               H, scale, window, stream))                                               \
      return rc;                                                                                                        \
    redo = 1;                                                                                                           \
  }
      KLLM_LATC(2, 6) KLLM_LATC(2, 8) KLLM_LATC(4, 10) KLLM_LATC(4, 12) KLLM_LATC(8, 18) KLLM_LATC(8, 20) KLLM_LATC(16, 34)
      KLLM_LATC(16, 36)
#undef KLLM_LATC
    }
    // the latent's accumulators and the query's pieces in registers: built for ranks up to 128, 256 and
    // 512 with rows of up to 256, 384 and 640; longer rows ask for the query at every tile
#define KLLM_LAT(NR, KS) launch_latent_mfma<NR, KS>(q, out, cache, positions, span_of_token, block_table, max_pages, page_size, n, H, row, rank, scale, window, part, nslices, redo, stream)
    if (rank <= 128) { if (row <= 256) KLLM_LAT(8, 8); else KLLM_LAT(8, 0); }
    else if (rank <= 256) { if (row <= 384) KLLM_LAT(16, 12); else KLLM_LAT(16, 0); }
    else { if (row <= 576) KLLM_LAT(32, 18); else if (row <= 640) KLLM_LAT(32, 20); else KLLM_LAT(32, 0); }
#undef KLLM_LAT
    KLLM_CHECK_LAUNCH("attn_latent");
    return 0;
  }
  if (dtype == DT_F32)
    hipLaunchKernelGGL(attn_latent_kernel<float>, dim3(n, H), dim3(kLatThreads), 0, stream, (const float*)q,
                       (float*)out, (const float*)cache, positions, span_of_token, block_table, max_pages, page_size, H,
                       row, rank, scale, window);
  else
    hipLaunchKernelGGL(attn_latent_kernel<bf16_t>, dim3(n, H), dim3(kLatThreads), 0, stream, (const bf16_t*)q,
                       (bf16_t*)out, (const bf16_t*)cache, positions, span_of_token, block_table, max_pages, page_size,
                       H, row, rank, scale, window);
  KLLM_CHECK_LAUNCH("attn_latent");
  return 0;
}

extern "C" int kllm_latent_out(const void* attended, const void* w_uv, const float* gate, int nsplit, long split_stride,
                               long gate_stride, void* out, int n, int H, int dv, int rank, int dtype, int gate_by_head,
                               hipStream_t stream) {
  KLLM_REQUIRE(attended && w_uv && out, "latent_out: null pointer");
  KLLM_REQUIRE(n > 0 && H > 0 && H <= 65535 && dv > 0 && rank > 0 && rank <= 8192 && (!gate || nsplit >= 1),
               "latent_out: bad sizes n=%d H=%d dv=%d rank=%d", n, H, dv, rank);
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "latent_out: unknown dtype %d", dtype);
  if (dtype == DT_BF16 && n >= kLatTokens && rank % 16 == 0 && ((uintptr_t)attended & 15) == 0 && ((uintptr_t)w_uv & 15) == 0 &&
      (n + kLatTokens - 1) / kLatTokens <= 65535 && (dv + 63) / 64 <= 65535) {
    const dim3 grid(H, (n + kLatTokens - 1) / kLatTokens, (dv + 127) / 128), halves(H, grid.y, (dv + 63) / 64);
#define KLLM_LOC(U, CHUNK, G)                                                                                                     \
  hipLaunchKernelGGL((latent_out_block_kernel<U, CHUNK>), G, dim3(kLatThreads), 0, stream, (const bf16_t*)attended, (const bf16_t*)w_uv, n, \
                     H, dv, rank, gate, gate_stride, nsplit, gate_by_head, split_stride, (bf16_t*)out)
#define KLLM_LO(U, G)                                                                                        \
  do {                                                                                                       \
    if (rank <= 128) KLLM_LOC(U, 128, G); else if (rank <= 256) KLLM_LOC(U, 256, G); else KLLM_LOC(U, 512, G); \
  } while (0)
    if (dv <= 64 || (long)H * grid.y * grid.z <= device_cus()) KLLM_LO(1, halves); else KLLM_LO(2, grid);
#undef KLLM_LO
#undef KLLM_LOC
    KLLM_CHECK_LAUNCH("latent_out");
    return 0;
  }
  if (dtype == DT_BF16 && rank % 32 == 0 && ((uintptr_t)attended & 15) == 0 && ((uintptr_t)w_uv & 15) == 0 && (dv + 15) / 16 <= 65535) {
    hipLaunchKernelGGL(latent_out_mfma_kernel, dim3((n + 15) / 16, H, (dv + 15) / 16), dim3(kWave), 0, stream, (const bf16_t*)attended,
                       (const bf16_t*)w_uv, n, H, dv, rank, gate, gate_stride, nsplit, gate_by_head, split_stride, (bf16_t*)out);
    KLLM_CHECK_LAUNCH("latent_out");
    return 0;
  }
  const size_t lds = (size_t)rank * sizeof(float);
  if (dtype == DT_F32)
    hipLaunchKernelGGL(latent_out_kernel<float>, dim3(n, H), dim3(kLatThreads), lds, stream, (const float*)attended,
                       (const float*)w_uv, gate, nsplit, split_stride, gate_stride, gate_by_head, (float*)out, H, dv, rank);
  else
    hipLaunchKernelGGL(latent_out_kernel<bf16_t>, dim3(n, H), dim3(kLatThreads), lds, stream, (const bf16_t*)attended,
                       (const bf16_t*)w_uv, gate, nsplit, split_stride, gate_stride, gate_by_head, (bf16_t*)out, H, dv, rank);
  KLLM_CHECK_LAUNCH("latent_out");
  return 0;
}
