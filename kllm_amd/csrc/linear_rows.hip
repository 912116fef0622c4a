// Products of up to 64 rows of X (decode batches, short prompts) on MFMA in bfloat16, with the step after
// the product in the same launch: the outputs of fused_linear.hpp, the weights in the lanes' order.
//
// What bounds such a product is the weights' way from memory and the rows' way from L2 into the CUs.  With tiles
// whose operands both pass through LDS (gemm_ring.hip) 64 rows are one row of tiles, K has to go in
// slices to fill the chip, and a second kernel adds the slices: norm, rotation and gate are launches of
// their own, about 4.7 us each at these sizes.  fused_linear.hip stages all rows in LDS first, and more than 32 rows of
// 2,048 do not fit.  Here nothing is staged: the waves of a workgroup share K, so no two of them want
// the same element of X, and each loads its fragments of the rows (from L2) and of the weights (from memory)
// straight into registers, four to eight steps of K in flight.  The waves meet once, when their sums
// are complete, and the epilogue runs on the whole sums.  (Sixteen waves, or twelve steps in flight: up to 30 % slower.)
//
// A workgroup owns TW tiles of 16 rows of W and NT tiles of 16 rows of X.  Every workgroup reads its rows
// of X whole, so TW is what divides the traffic from L2.  Two workgroups may share a tile of W and take half of the rows each;
// they sit on one XCD, so that the weights come from memory once.
//
// Rows that go from one such product to the next are stored in the order its lanes read (rows_at): a load is then one contiguous
// kilobyte, or less where there are fewer rows than 16.  From rows as they are, its sixteen lanes with one K lie in sixteen
// rows, and a CU takes in 16 bytes a clock (64 rows of 5,632 against 2,048 columns: 15.8 -> 12.1 us; 16 rows 11.2 -> 10.1).
//
// At a few rows a launch is mostly its own beginning and end: of 4.9 us for 2,048 x 2,048 at one row the weights take 1.6.  So what the
// loads of the weights need comes with the launch (the first fourteen words of the arguments lie in scalar registers when a wave starts; a trip
// to the arguments is 0.3 us in a cold cache, and there were three in a row), they are the first thing that a wave asks for, and
// what only the epilogue needs comes behind them.
//
// Alone in a replayed graph, 1 / 8 / 16 / 64 rows (tiled, but for 2,048 x 2,048), us, before that and now: 2,048 x 2,048 4.9 / 5.8 /
// 7.3 / 7.7, 3.7 / 4.2 / 5.0 / 7.0; 2,048 x 5,632 7.5 / 8.0 / 9.4 / 12.0, 6.4 / 6.8 / 8.0 / 11.2; 2 x 5,632 x 2,048 10.9 / 11.0 / 11.3 / 14.1, 10.1 /
// 10.2 / 10.6 / 13.9; plain sums 2,560 x 2,048 4.6 / 4.8 / 5.2 / 8.6, 3.9 / 4.2 / 4.5 / 8.0; 4,096 x 4,096 8.9 / 9.2 / 9.3 / 14.6, 7.9 / 8.1 / 8.3
// / 13.8; 4,096 x 14,336 23.5 / 24.1 / 25.9 / 44.7, 22.8 / 23.1 / 25.0 / 42.6 (117 MB: 5.1 TB/s).  A decode step at 1.1B sizes, 1 / 8 / 64 tokens
// 874 / 945 / 1,575 -> 794 / 868 / 1,530 us, 45 tokens of prompt 1,027 -> 958, 8B sizes at 16 tokens 3,980 -> 3,855, float32 at 8 1,565 -> 1,510.
#include <math.h>

#include "common.hpp"
#include "fused_linear.hpp"
#include "kllm_kernels.h"

namespace kllm {

typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr int LR_ROWS = 64;             // rows of X at most
constexpr int LR_LD = 20;               // floats from one x row of a partial tile to the next: 16 and padding, whole 16 bytes
constexpr int LR_TILE = 16 * LR_LD;

// Steps of K in each of the two buffers a wave fills in turn: what 128 registers hold, four at most.
constexpr int lr_ahead(int nt, int tw) { return nt + tw <= 4 ? 4 : nt + tw == 5 ? 3 : 2; }

// A: steps of K in each of the two buffers.
// SPLIT (FL_RESID and FL_PARTS, up to 16 rows): a workgroup takes eight rows of W, each twice in a matrix instruction: K's first half in its rows
// 0-7, the second half in rows 8-15, so that a load still brings a kilobyte.  Up to eight rows of X lie in the operand's columns the
// same way (NT 1); more take an instruction for each half of K (NT 2).  What pairs a half with the other's X is not used.  A CU streams
// about 20 GB/s of weights from memory whatever a workgroup has in flight, so a product on half the CUs takes half as long again:
// a step at 1.1B sizes, 1 / 8 / 16 tokens 894 / 939 / 1,032 us without, 882 / 920 / 1,026 with.
// float32 (up to 16 rows): four instructions of 4 to a step, true 32-bit.  A sum's products go in 64 or 128 chains, no fewer than in the
// decode-batch kernel: 16 a wave, or 8 where eight waves take the place of its four (the gate, plain sums).
template <typename T, int EP> constexpr int lr_chains() { return sizeof(T) == 2 ? 1 : EP == FL_RESID || EP == FL_ROPE ? 16 : 8; }
__device__ __forceinline__ void lr_mma(uintx4 w, uintx4 x, floatx4 (&acc)[1], int, bf16_t) {
  acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), acc[0], 0, 0, 0);
}
template <int CH>
__device__ __forceinline__ void lr_mma(uintx4 w, uintx4 x, floatx4 (&acc)[CH], int i, float) {
  const floatx4 a = __builtin_bit_cast(floatx4, w), b = __builtin_bit_cast(floatx4, x);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    floatx4& c = acc[(4 * i + e) % CH];
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  }
}

enum : unsigned { LR_HALVES = 1, LR_X_TILED = 2, LR_W_TILED = 4 };

template <typename T, int NT, int TW, int EP, bool SCALED, int NW, bool SPLIT, int A>
__global__ __launch_bounds__(64 * NW) void linear_rows_kernel(const T* __restrict__ W, const T* __restrict__ X, int m, int k,
                                                              int x_stride, unsigned how, const int* __restrict__ positions,
                                                              const int* __restrict__ span_of_token, const float* __restrict__ ss_in,
                                                              FlOut out) {
  const int n = how >> 8 & 0xFF, ss_parts = how >> 16;
  constexpr int ES = (int)sizeof(T), CH = lr_chains<T, EP>();    // (n and ss_parts share a word with the flags: all of it in fourteen)
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  float* part = reinterpret_cast<float*>(lds_raw);               // [NW][TW][NT][x row 16][LR_LD]
  float* row_scale = part + NW * TW * NT * LR_TILE;              // [16 NT]
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane / 16, c = lane % 16;
  const int tiles = EP == FL_RESID || EP == FL_PARTS ? (int)((unsigned)(m + 15) / 16) : (int)((unsigned)(m / 2 + 7) / 8);
  const int groups = (int)((unsigned)(tiles + TW - 1) / TW);     // workgroups side by side over W
  const bool halved = how & LR_HALVES;
  // Blocks go to the XCDs in turn: two workgroups of one group of tiles are eight blocks apart.
  const int group = SPLIT ? (int)(blockIdx.x / 2) : !halved ? (int)blockIdx.x : (int)(blockIdx.x / 16) * 8 + (int)(blockIdx.x % 8);
  const int half_tile = SPLIT ? (int)(blockIdx.x % 2) : 0;       // which eight rows of W
  const int row0 = halved ? (int)(blockIdx.x / 8 % 2) * (16 * NT) : 0;
  if (group >= groups || row0 >= n) return;                      // the whole workgroup
  const int steps = (int)((unsigned)k / (64 / ES));              // of 64 bytes of a row (k is a multiple of 32)
  const int walk = SPLIT ? steps / 2 : steps;                    // steps that the waves share
  const int per = (int)((unsigned)(walk + NW - 1) / NW);
  const int s_beg = min(wave * per, walk);
  const int mine = min(per, walk - s_beg);                       // steps of this wave, possibly none

  // ---- loads return in order: a rotation's page takes two trips, so its position goes first, and so do the sums of squares,
  // which are added while the weights are on their way (behind the weights: up to 3 % of a step slower)
  const int half = EP == FL_ROPE ? out.hd / 2 : 1;
  constexpr int RC = SPLIT ? 8 : 16;                             // columns of a workgroup's output tile, and threads to a row
  constexpr int RR = 64 * NW / RC;                               // rows that the threads take at a time
  constexpr int RU = ((SPLIT ? 16 : 16 * NT) + RR - 1) / RR;                    // turns
  constexpr int PU = EP == FL_ROPE ? (16 * NT + 2 * RR - 1) / (2 * RR) : 1;
  int ep_pos[PU], ep_span[PU], ep_page[PU];
  if (EP == FL_ROPE) {         // thread (pair tid % 8, row tid / 8, and 2 RR on)
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int xr = min(row0 + tid / 8 + 2 * RR * u, n - 1);
      ep_pos[u] = positions ? positions[xr] : 0;
      ep_span[u] = positions ? span_of_token[xr] : 0;
    }
  }

  // ---- operands: offsets in bytes from descriptors that all lanes share, so that a step costs a scalar
  // addition; the weights of a buffer before its rows, which come from nearer.  A step that does not exist reads the wave's last (or K's last) again and is not multiplied; a
  // tile or a row of X beyond the last one reads the last, and its sums are not stored.
  const int tile0 = group * TW;
  // (float32 also takes the weights as they are, row by row: the sums are the same bits, so that a card with no room for
  // the tiled copy gives the same results)
  const bool tiled = ES == 2 || (how & LR_W_TILED), x_tiled = how & LR_X_TILED;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(W)) + (tiled ? (long)tile0 * steps * 1024 : 0), 0,
      tiled ? min(TW, tiles - tile0) * steps * 1024 : m * k * ES, 0x00020000);
  const int w_step = tiled ? 1024 : 64;
  const int later = SPLIT && c >= 8 ? walk : 0;                  // steps on, for the lanes of the second half of K
  const int wc = SPLIT ? 8 * half_tile + c % 8 : c;              // this lane's row of a tile
  int wo[TW], xo[NT];
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    const int tile = min(j, tiles - tile0 - 1);
    wo[j] = tile * steps * 1024 + later * 1024 + (16 * g + wc) * 16;
    if (!tiled) wo[j] = (int)max(fl_row<EP>(tile0 + tile, wc, m, out), 0L) * k * ES + later * 64 + 16 * g;
  }
  const int s_last = min(s_beg + max(mine, 1), walk) - 1;
  auto fill_w = [&](uintx4 (&wb)[A][TW], int s0) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
        wb[i][j] = __builtin_amdgcn_raw_buffer_load_b128(wr, wo[j], min(s_beg + s0 + i, s_last) * w_step, 0);
  };
  const int row_tiles = (n + 15) / 16, side = min(n, 16), x_step = x_tiled ? 64 * side : 64;
  const __amdgpu_buffer_rsrc_t xr_ = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(X), 0, x_tiled ? row_tiles * steps * x_step : ES * ((n - 1) * x_stride + k), 0x00020000);
#pragma unroll
  for (int t = 0; t < NT; ++t)
    xo[t] = x_tiled ? min(row0 / 16 + t, row_tiles - 1) * steps * x_step + (g * side + min(c, side - 1)) * 16
                    : ES * min(row0 + t * 16 + c, n - 1) * x_stride + 16 * g;
  if (SPLIT) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = min(NT == 1 ? c % 8 : c, n - 1);
      xo[t] = (NT == 1 ? later : t * walk) * x_step + (x_tiled ? (g * side + row) * 16 : ES * row * x_stride + 16 * g);
    }
  }
  auto fill_x = [&](uintx4 (&xb)[A][NT], int s0) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        xb[i][t] = __builtin_amdgcn_raw_buffer_load_b128(xr_, xo[t], min(s_beg + s0 + i, s_last) * x_step, 0);
  };
  auto fill = [&](uintx4 (&wb)[A][TW], uintx4 (&xb)[A][NT], int s0) {
    fill_w(wb, s0);
    fill_x(xb, s0);
    // Loads and products stay on their sides of this line: left to itself the compiler moves half of the
    // loads to where their values are used.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  floatx4 acc[TW][NT][CH];
#pragma unroll
  for (int j = 0; j < TW; ++j)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < CH; ++e) acc[j][t][e] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](const uintx4 (&wb)[TW], const uintx4 (&xb)[NT], int i) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < TW; ++j) lr_mma(wb[j], xb[t], acc[j][t], i, T());
  };
  // (whole words: as bfloat16 vectors the compiler puts the halves together again behind each load, and waits for it)
  uintx4 wa[A][TW], xa[A][NT], wb[A][TW], xb[A][NT];
  constexpr int SU = RU;
  floatx4 ssv[SCALED ? SU : 1][FL_SS_LOADS];
  if (SCALED) {
    const int stride = (ss_parts + 3) / 4 * 4;
#pragma unroll
    for (int u = 0; u < SU; ++u)
#pragma unroll
      for (int i = 0; i < FL_SS_LOADS; ++i) {
        const int at = 4 * (tid % 16 + 16 * i);
        ssv[u][i] = *reinterpret_cast<const floatx4*>(ss_in + (long)min(row0 + tid / 16 + RR * u, n - 1) * stride +
                                                      (at < stride ? at : 0));
      }
  }
  fill(wa, xa, 0);
  // ---- what the epilogue needs: behind the first operands
  float ep_cos[PU], ep_sin[PU], res_old[RU], res_w = 0.f;
  if (EP == FL_ROPE) {
    const int pair = group * 8 + tid % 8;
    const bool turns = out.cos_t && pair < (out.H + (out.cache ? out.KV : 0)) * half;
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int xr = min(row0 + tid / 8 + 2 * RR * u, n - 1);
      ep_cos[u] = turns ? out.cos_t[(long)xr * half + pair % half] : 1.f;
      ep_sin[u] = turns ? out.sin_t[(long)xr * half + pair % half] : 0.f;
      ep_page[u] = out.cache ? out.block_table[(long)ep_span[u] * out.max_pages + ep_pos[u] / out.page_size] : 0;
    }
  }
  if (SCALED) {      // the rows' scales, before the second buffer needs the registers: sums in a fixed order, then across sixteen lanes
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < FL_SS_LOADS; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) v += 4 * (tid % 16 + 16 * i) + e < ss_parts ? ssv[u][i][e] : 0.f;
      v = parts_sum<16>(v);
      if (tid % 16 == 0 && tid / 16 + RR * u < 16 * NT) row_scale[tid / 16 + RR * u] = rsqrtf(v / (float)k + out.eps);
    }
  }
  auto ask_stream = [&] {
    if (EP != FL_RESID) return;  // thread (w row tid % RC, x row tid / RC and RR on)
    const int col = min(group * 16 + 8 * half_tile + tid % RC, m - 1);
    res_w = out.norm_w[col];
#pragma unroll
    for (int u = 0; u < RU; ++u) res_old[u] = out.resid[(long)min(row0 + tid / RC + RR * u, n - 1) * m + col];
  };
  if (SPLIT && ES == 2 && per <= A) {      // (K of up to 2,048: one buffer is all a wave has)
    ask_stream();
#pragma unroll
    for (int i = 0; i < A; ++i)
      if (i < mine) step(wa[i], xa[i], i);
  } else {
    fill(wb, xb, A);
    ask_stream();
    int s = 0;
    for (; mine - s > 2 * A; s += 2 * A) {
#pragma unroll
      for (int i = 0; i < A; ++i) step(wa[i], xa[i], i);
      __builtin_amdgcn_sched_barrier(0);
      fill(wa, xa, s + 2 * A);
#pragma unroll
      for (int i = 0; i < A; ++i) step(wb[i], xb[i], i);
      __builtin_amdgcn_sched_barrier(0);
      fill(wb, xb, s + 3 * A);
    }
#pragma unroll
    for (int i = 0; i < A; ++i)
      if (s + i < mine) step(wa[i], xa[i], i);
#pragma unroll
    for (int i = 0; i < A; ++i)
      if (s + A + i < mine) step(wb[i], xb[i], i);
  }

  // ---- the waves meet: lane (g, c) holds w rows 4 g ... 4 g + 3 of x row c
#pragma unroll
  for (int j = 0; j < TW; ++j)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int d = CH / 2; d > 0; d >>= 1)                       // (the chains, in pairs)
#pragma unroll
        for (int e = 0; e < d; ++e) acc[j][t][e] += acc[j][t][e + d];
      *reinterpret_cast<floatx4*>(&part[((wave * TW + j) * NT + t) * LR_TILE + c * LR_LD + 4 * g]) = acc[j][t][0];
    }
  fl_lds_barrier();
  auto sum_of = [&](int j, int t, int xc, int r) {               // in pairs
    float v[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* of = part + ((w * TW + j) * NT + t) * LR_TILE + xc * LR_LD + r;
      v[w] = of[0];
      if (SPLIT) v[w] += NT == 1 ? of[8 * LR_LD + 8] : of[LR_TILE + 8];    // the second half of K
    }
#pragma unroll
    for (int d = NW / 2; d > 0; d >>= 1)
#pragma unroll
      for (int w = 0; w < d; ++w) v[w] += v[w + d];
    return v[0];
  };
  if (EP == FL_RESID) {
    const int col = group * 16 + 8 * half_tile + tid % RC;
    const int parts = SPLIT ? 2 * groups : groups, stride = (parts + 3) / 4 * 4;
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int r = tid / RC + RR * u, xr = row0 + r;
      const bool live = r < 16 * NT && xr < n && col < m;
      float x = 0.f;
      if (live) {
        x = res_old[u] + sum_of(0, SPLIT ? 0 : r / 16, r % 16, tid % RC);
        out.resid[(long)xr * m + col] = x;
        reinterpret_cast<T*>(out.y)[rows_at(out.y_tiled ? min(n, 16) : 0, xr, col, m)] = from_f32<T>(x * res_w);
      }
      const float ss = parts_sum<RC>(x * x);
      if (tid % RC == 0 && r < 16 * NT && xr < n) out.ss_out[(long)xr * stride + (SPLIT ? (int)blockIdx.x : group)] = ss;
    }
    return;
  }
  if (EP == FL_PARTS) {                // the sums, or an activation of them in 16 bits
    constexpr int C = SPLIT ? 8 : 16 * TW, ROWS = SPLIT ? 16 : 16 * NT;
#pragma unroll 1
    for (int u = 0; u < (ROWS * C + 64 * NW - 1) / (64 * NW); ++u) {
      const int idx = tid + 64 * NW * u;
      const int cc = idx % C, r = idx / C, xr = row0 + r, col = group * (16 * TW) + 8 * half_tile + cc;
      if (r >= ROWS || xr >= n || col >= m) continue;
      const float v = sum_of(SPLIT ? 0 : cc / 16, SPLIT ? 0 : r / 16, r % 16, SPLIT ? cc : cc % 16);
      if (out.act >= FL_UNARY) {
        float a_pos = 0.f, a_neg = 0.f;
        if (out.act - FL_UNARY == ACT_XIELU) {
          a_pos = softplus_f32(out.norm_w[0]);
          a_neg = softplus_f32(out.norm_w[1]);
        }
        reinterpret_cast<T*>(out.y)[(long)xr * m + col] = from_f32<T>(unary_act<T>(v, out.act - FL_UNARY, a_pos, a_neg));
      } else {
        reinterpret_cast<float*>(out.y)[(long)xr * m + col] = v;
      }
    }
    return;
  }
  if (EP == FL_SWIGLU || EP == FL_ROPE) {
    constexpr int P = 8 * TW;                                    // pairs of a row in the workgroup
    const int pairs = m / 2;
    auto pair_out = [&](int u) {
      const int idx = tid + 64 * NW * u;
      const int p = idx % P, r = idx / P, xr = row0 + r, pair = group * P + p;
      if (r >= 16 * NT || pair >= pairs || xr >= n) return;
      float a = sum_of(p / 8, r / 16, r % 16, p % 8), b = sum_of(p / 8, r / 16, r % 16, p % 8 + 8);
      if (SCALED) {
        a *= row_scale[r];
        b *= row_scale[r];
      }
      if (EP == FL_SWIGLU) {
        reinterpret_cast<T*>(out.y)[rows_at(out.y_tiled ? min(n, 16) : 0, xr, pair, pairs)] = from_f32<T>(gate_act<T>(a, out.act) * b);
      } else {
        const int e = EP == FL_ROPE ? u : 0;
        fl_rope_store<T>(out, xr, pair, a, b, ep_cos[e], ep_sin[e], ep_page[e], out.cache ? ep_pos[e] % out.page_size : 0);
      }
    };
    if (EP == FL_ROPE) {
#pragma unroll
      for (int u = 0; u < PU; ++u) pair_out(u);
    } else {                           // (one copy of the code: it is read cold at every launch)
#pragma unroll 1
      for (int u = 0; u < (16 * NT * P + 64 * NW - 1) / (64 * NW); ++u) pair_out(u);
    }
  }
}

static size_t lr_lds_bytes(int nt, int tw, int nw) { return (size_t)(nw * tw * nt * LR_TILE + LR_ROWS) * sizeof(float); }

template <typename T, int NT, int TW, int EP, bool SCALED, int NW, bool SPLIT = false, int A = lr_ahead(NT, TW)>
static int lr_launch_waves(const void* x, const FlOut& out, const void* w, int n, int m, int k, int tiles, int halves,
                     int x_stride, hipStream_t stream) {
  const size_t lds = lr_lds_bytes(NT, TW, NW);
  if (lds > 64 * 1024) {
    static const hipError_t e = hipFuncSetAttribute((const void*)linear_rows_kernel<T, NT, TW, EP, SCALED, NW, SPLIT, A>,
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) KLLM_FAIL((int)e, "linear_rows: cannot raise the LDS limit: %s", hipGetErrorString(e));
  }
  const int groups = ceil_div(tiles, TW);
  const int blocks = SPLIT ? 2 * groups : halves == 1 ? groups : ceil_div(groups, 8) * 16;
  hipLaunchKernelGGL((linear_rows_kernel<T, NT, TW, EP, SCALED, NW, SPLIT, A>), dim3(blocks), dim3(64 * NW), lds, stream,
                     (const T*)w, (const T*)x, m, k, x_stride,
                     (halves == 2 ? LR_HALVES : 0u) | (out.x_tiled ? LR_X_TILED : 0u) | (out.tiled ? LR_W_TILED : 0u) |
                         (unsigned)n << 8 | (unsigned)out.ss_parts << 16,
                     out.cache ? out.positions : nullptr, out.cache ? out.span_of_token : nullptr, out.ss_in, out);
  return 0;
}

template <typename T, int NT, int TW, int EP, bool SCALED>
static int lr_launch(const void* x, const FlOut& out, const void* w, int n, int m, int k, int tiles, int halves,
                     int x_stride, hipStream_t stream) {
  // Four waves a workgroup where a CU has several of them (4,096 -> 6,144: 14.7 us with eight, 13.3 with four), eight where it
  // has one (a step of one token at 1.1B sizes 0.3 % shorter, of 64 tokens 1.2 %).
  if constexpr ((EP != FL_SWIGLU && EP != FL_PARTS) || (TW == 3 && sizeof(T) == 2))
    if ((long)halves * ceil_div(tiles, TW) > device_cus())
      return lr_launch_waves<T, NT, TW, EP, SCALED, 4>(x, out, w, n, m, k, tiles, halves, x_stride, stream);
  return lr_launch_waves<T, NT, TW, EP, SCALED, 8>(x, out, w, n, m, k, tiles, halves, x_stride, stream);
}

template <typename T, int NT, int TW>
static int lr_launch_ep(int ep, bool scaled, const void* x, const FlOut& out, const void* w, int n, int m, int k,
                        int tiles, int halves, int xs, hipStream_t st) {
  if (ep == FL_SWIGLU)
    return scaled ? lr_launch<T, NT, TW, FL_SWIGLU, true>(x, out, w, n, m, k, tiles, halves, xs, st)
                  : lr_launch<T, NT, TW, FL_SWIGLU, false>(x, out, w, n, m, k, tiles, halves, xs, st);
  if (ep == FL_PARTS) return lr_launch<T, NT, TW, FL_PARTS, false>(x, out, w, n, m, k, tiles, halves, xs, st);
  if constexpr (TW == 1) {
    if (ep == FL_RESID) return lr_launch<T, NT, 1, FL_RESID, false>(x, out, w, n, m, k, tiles, halves, xs, st);
    return scaled ? lr_launch<T, NT, 1, FL_ROPE, true>(x, out, w, n, m, k, tiles, halves, xs, st)
                  : lr_launch<T, NT, 1, FL_ROPE, false>(x, out, w, n, m, k, tiles, halves, xs, st);
  }
  KLLM_FAIL(ERR_STATE, "linear_rows: no kernel for output kind %d and %d tiles", ep, TW);
}

template <typename T, int NT>
static int lr_launch_tw(int tw, int ep, bool scaled, const void* x, const FlOut& out, const void* w, int n, int m, int k,
                        int tiles, int halves, int xs, hipStream_t st) {
  if (tw == 1) return lr_launch_ep<T, NT, 1>(ep, scaled, x, out, w, n, m, k, tiles, halves, xs, st);
  if (tw == 2) return lr_launch_ep<T, NT, 2>(ep, scaled, x, out, w, n, m, k, tiles, halves, xs, st);
  return lr_launch_ep<T, NT, 3>(ep, scaled, x, out, w, n, m, k, tiles, halves, xs, st);
}

}  // namespace kllm

using namespace kllm;

static int lr_tiles(int kind, int m) { return kind == FL_RESID || kind == FL_PARTS ? ceil_div(m, 16) : ceil_div(m / 2, 8); }

// Whether a product that splits takes eight rows of W a workgroup (SPLIT): up to 16 rows of X and no more tiles than half the CUs.
static bool lr_split(int n, int m, int k) { return n <= 16 && k % 64 == 0 && 2 * lr_tiles(FL_RESID, m) <= device_cus(); }

// Whether a SPLIT product's waves fill their buffers three steps at a time instead of four: a wave asks for whole turns of both
// buffers, and what is beyond its last step is read again for nothing.  2,048 x 5,632 (eleven steps a wave, sixteen asked
// for in fours, twelve in threes), 1 / 8 rows alone in a replayed graph: 6.7 / 8.2 us in fours, 6.5 / 7.5 in threes, 6.4 / 7.7 in sixes;
// 2,048 x 2,048 (four steps: one buffer) 3.6 / 4.2, 3.8 / 4.7, 3.8 / 4.5.
static bool lr_threes(int k) {
  const int per = ceil_div(k / 64, 8);
  return per > 4 && ceil_div(per, 6) * 6 < ceil_div(per, 8) * 8;
}

// Tiles of W a workgroup, workgroups that share the rows out, tiles of rows a workgroup.
struct LrPlan {
  int tw, halves, nt;
};

static LrPlan lr_plan(int ep, int n, int m, int k, bool f32, bool x_tiled) {
  const int cus = device_cus(), tiles = lr_tiles(ep, m);
  LrPlan p = {1, 1, ceil_div(n, 16)};
  if (ep == FL_SWIGLU || ep == FL_PARTS) {
    // Tiles a workgroup: the least that leaves one round of the chip, three at most (2 x 5,632 x 2,048, 8 / 64 rows: 12.1 / 17.5 us with two, 11.0
    // / 14.9 with three, 13.3 / 16.4 with four; 2 x 14,336 x 4,096, 16 / 64 rows: 48.5 / 62.0, 46.5 / 59.3, 54.5 / 59.6).
    while (p.tw < 3 && ceil_div(tiles, p.tw) > cus) ++p.tw;
    // Many rounds: one tile, of which a CU holds two workgroups, where K is long; two where a workgroup is short, or where many
    // rows that lie as they are (slow to read) are read once for both.  us with one / two / three: 2 x 14,336 x 4,096, 8 rows 41.4 / 45.6 / 45.9, 16 rows
    // 45.2 / 47.0 / 47.5, as they are 9 42.0 / 46.6, 12 44.5 / 46.4, 16 49.1 / 46.8 / 48.3; 2 x 13,824 x 5,120, 12 rows as they are 61.7 / 57.8 / 58.9; 2 x 8,192 x 3,072, 16 rows 23.4 / 20.9 / 23.7; x 2,048, 1 row
    // 13.7 / 14.1 / 15.6; 2 x 11,008 x 1,024, 8 rows 14.0 / 11.9 / 10.5.  float32, whose rows are as they are: 2 x 8,192 x 2,048, 8 / 16 rows 25.6
    // / 29.9 with one, 28.5 / 29.2 with two; 2 x 7,168 x 1,536 21.5 / 26.6, 21.3 / 23.6.
    if (tiles > 3 * cus) p.tw = n > 16 ? 1 : n <= 8 ? (f32 || k >= 2048 ? 1 : 2) : f32 ? (k >= 2048 ? 1 : 2) : (k >= 4096 && (x_tiled || n * k <= 49152) ? 1 : 2);
  }
  // Halves of the rows where the busiest CU then has fewer tiles of rows to take (or as many, of workgroups that share it
  // anyway): 64 rows against 2,048 x 5,632 (128 tiles) 17.6 -> 12.2 us, 6,144 x 4,096 (384) 25.4 -> 21.2, 48 rows 21.3 -> 18.8; not
  // 4,096 x 14,336 (256) 41.0 -> 46.7, nor 2,560 x 2,048 (160) at 32 rows 5.0 -> 5.5.
  const int whole = ceil_div(tiles, cus) * p.nt, halved = ceil_div(2L * tiles, cus) * ceil_div(p.nt, 2);
  if (ep != FL_SWIGLU && p.tw == 1 && (halved < whole || (halved == whole && tiles > cus))) {
    p.halves = 2;
    p.nt = ceil_div(p.nt, 2);
  }
  return p;
}

extern "C" int kllm_linear_rows_row_tiles(int kind, int n, int m, int k) {
  if (n <= 0 || m <= 0 || k <= 0) return 0;
  const LrPlan p = lr_plan(kind, n, m, k, false, true);
  return ceil_div((long)ceil_div(lr_tiles(kind, m), p.tw) * p.halves, device_cus()) * p.nt;
}

extern "C" int kllm_linear_rows_parts(int n, int m, int k) {
  if (n <= 0 || m <= 0 || k <= 0) return 0;
  const int parts = lr_split(n, m, k) ? 2 * lr_tiles(FL_RESID, m) : lr_tiles(FL_RESID, m);
  return parts <= FL_SS_MAX ? parts : 0;
}

extern "C" int kllm_linear_rows(const void* x, int x_stride, const KllmLinearOut* yout, const void* w, int n, int m, int k,
                                hipStream_t stream) {
  KLLM_REQUIRE(x && yout && w && yout->y, "linear_rows: null pointer");
  const int ep = yout->kind;
  KLLM_REQUIRE(ep == FL_PARTS || ep == FL_RESID || ep == FL_SWIGLU || ep == FL_ROPE, "linear_rows: unknown output kind %d", ep);
  const bool f32 = yout->f32 != 0;
  KLLM_REQUIRE(n > 0 && n <= (f32 ? 16 : LR_ROWS), "linear_rows: n=%d is outside [1, %d]", n, f32 ? 16 : LR_ROWS);
  KLLM_REQUIRE(m > 0 && k > 0 && k % 32 == 0, "linear_rows: bad sizes m=%d k=%d (K must be a multiple of 32)", m, k);
  KLLM_REQUIRE(k <= (1 << 20) && m < (1 << 30), "linear_rows: sizes overflow");
  KLLM_REQUIRE((yout->tiled || f32) && yout->nsplit <= 1, "linear_rows: takes the tiled copy of the weights and all of K");
  KLLM_REQUIRE(yout->tiled || (long)m * k < (1L << 29), "linear_rows: %d x %d weights need their tiled copy", m, k);
  KLLM_REQUIRE(!f32 || (!yout->x_tiled && !yout->y_tiled), "linear_rows: tiled rows are bfloat16");
  KLLM_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "linear_rows: operands must be 16-byte aligned");
  if (x_stride <= 0) x_stride = k;
  KLLM_REQUIRE(x_stride >= k && x_stride % (f32 ? 4 : 8) == 0 && x_stride < (1 << 23), "linear_rows: row stride %d of x does not fit K=%d",
               x_stride, k);
  FlOut out = {};
  out.y = yout->y;
  out.act = yout->act;
  out.tiled = yout->tiled ? 1 : 0;
  out.x_tiled = yout->x_tiled != 0;
  out.y_tiled = yout->y_tiled != 0;
  KLLM_REQUIRE(!out.y_tiled || (ep == FL_RESID && m % 32 == 0) || (ep == FL_SWIGLU && m % 64 == 0),
               "linear_rows: no tiled output of kind %d and m=%d", ep, m);
  const int tiles = lr_tiles(ep, m);
  const bool scaled = yout->ss_in != nullptr;
  if (scaled) {
    KLLM_REQUIRE(ep != FL_RESID && ep != FL_PARTS, "linear_rows: only the gate and the rotation epilogues scale their rows");
    KLLM_REQUIRE(yout->ss_parts >= 1 && yout->ss_parts <= FL_SS_MAX && ((uintptr_t)yout->ss_in & 15) == 0 && yout->eps >= 0.f,
                 "linear_rows: %d partial sums of squares per row are outside [1, %d], or they are not 16-byte aligned",
                 yout->ss_parts, FL_SS_MAX);
    out.ss_in = yout->ss_in;
    out.ss_parts = yout->ss_parts;
    out.eps = yout->eps;
  }
  if (ep == FL_RESID) {
    KLLM_REQUIRE(yout->resid && yout->norm_w && yout->ss_out, "linear_rows: the residual epilogue needs the stream, "
                 "the norm's weight and room for the sums of squares");
    KLLM_REQUIRE(kllm_linear_rows_parts(n, m, k) > 0, "linear_rows: %d columns leave more than %d sums of squares per row", m,
                 FL_SS_MAX);
    out.resid = yout->resid;
    out.norm_w = yout->norm_w;
    out.ss_out = yout->ss_out;
  } else if (ep == FL_PARTS) {
    KLLM_REQUIRE(out.act < FL_UNARY + UNARY_ACT_COUNT, "linear_rows: unknown activation %d on the sums", out.act - FL_UNARY);
    KLLM_REQUIRE(out.act - FL_UNARY != ACT_XIELU || yout->norm_w, "linear_rows: this activation needs its two constants");
    out.norm_w = yout->norm_w;
  } else {
    KLLM_REQUIRE(m % 2 == 0, "linear_rows: m=%d must be even for a pair epilogue", m);
  }
  KLLM_REQUIRE(ep != FL_SWIGLU || (out.act >= 0 && out.act < ACT_COUNT), "linear_rows: unknown activation %d", out.act);
  if (ep == FL_ROPE) {
    const int H = yout->H, KV = yout->KV, hd = yout->hd;
    KLLM_REQUIRE(H > 0 && hd > 0 && hd % 2 == 0, "linear_rows: bad heads H=%d hd=%d", H, hd);
    KLLM_REQUIRE((yout->cos_t == nullptr) == (yout->sin_t == nullptr), "linear_rows: cos and sin go together");
    if (yout->cache)
      KLLM_REQUIRE(KV > 0 && yout->positions && yout->span_of_token && yout->block_table && yout->max_pages > 0 &&
                       yout->page_size > 0,
                   "linear_rows: bad cache arguments");
    KLLM_REQUIRE(m == H * hd + (yout->cache ? 2 * KV * hd : 0), "linear_rows: m=%d does not fit the heads", m);
    out.cos_t = yout->cos_t;
    out.sin_t = yout->sin_t;
    out.cache = yout->cache;
    out.positions = yout->positions;
    out.span_of_token = yout->span_of_token;
    out.block_table = yout->block_table;
    out.max_pages = yout->max_pages;
    out.page_size = yout->page_size;
    out.H = H;
    out.KV = KV;
    out.hd = hd;
  }
  const LrPlan plan = lr_plan(ep, n, m, k, f32, out.x_tiled);
  const int tw = plan.tw, halves = plan.halves, nt = plan.nt;
#define KLLM_LRS(NT, EP)                                                                                        \
  (f32           ? lr_launch_waves<float, NT, 1, EP, false, 8, true>(x, out, w, n, m, k, tiles, 1, x_stride, stream)       \
   : lr_threes(k) ? lr_launch_waves<bf16_t, NT, 1, EP, false, 8, true, 3>(x, out, w, n, m, k, tiles, 1, x_stride, stream)   \
                 : lr_launch_waves<bf16_t, NT, 1, EP, false, 8, true, 4>(x, out, w, n, m, k, tiles, 1, x_stride, stream))
  const bool split = (ep == FL_RESID || ep == FL_PARTS) && lr_split(n, m, k);
  const int rc = split     ? (ep == FL_RESID ? (n <= 8 ? KLLM_LRS(1, FL_RESID) : KLLM_LRS(2, FL_RESID))
                                             : (n <= 8 ? KLLM_LRS(1, FL_PARTS) : KLLM_LRS(2, FL_PARTS)))
               : f32     ? lr_launch_tw<float, 1>(tw, ep, scaled, x, out, w, n, m, k, tiles, 1, x_stride, stream)
               : nt == 1 ? lr_launch_tw<bf16_t, 1>(tw, ep, scaled, x, out, w, n, m, k, tiles, halves, x_stride, stream)
               : nt == 2 ? lr_launch_tw<bf16_t, 2>(tw, ep, scaled, x, out, w, n, m, k, tiles, halves, x_stride, stream)
               : nt == 3 ? lr_launch_tw<bf16_t, 3>(tw, ep, scaled, x, out, w, n, m, k, tiles, halves, x_stride, stream)
                         : lr_launch_tw<bf16_t, 4>(tw, ep, scaled, x, out, w, n, m, k, tiles, halves, x_stride, stream);
#undef KLLM_LRS
  if (rc) return rc;
  KLLM_CHECK_LAUNCH("linear_rows");
  return 0;
}
