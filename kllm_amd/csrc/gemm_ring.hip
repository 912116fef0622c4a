// Matrix products on MFMA tiles: Y[n, m] = X[n, k] . W[m, k]^T, bfloat16, or float32 in true 32-bit; prompts,
// and decode batches of more than 16 rows.
//
// One workgroup of eight waves a CU and output tile (256 x 256, 256 x 192 or 128 x 256; two or three
// workgroups a CU for smaller ones).  A tile's rows of X and of W come in two halves each; a stage
// is whole cache lines of K (128 bytes: 64 bfloat16 or 32 float32), so a stage is four sub-tiles, X0 X1 W0 W1, and LDS holds
// two stages of them: a ring of eight buffers.
//
// What bounds a kernel of this kind is the way from memory into LDS: with two whole stages that are
// filled, waited for and read one after the other, a CU has one stage in flight for one stage's
// time and waits for the rest (2,048 x 28,672 x 4,096: 499 us, matrix units busy 36 %).  Here a
// wave multiplies one quarter of its output at a time, a phase: (X0 W0) (X0 W1) (X1 W1) (X1 W0),
// the next stage in the mirrored order (X0 W1) (X0 W0) (X1 W0) (X1 W1).  Every phase then reads
// exactly one new sub-tile from LDS (the other operand is in registers already), which frees
// its buffer at once, and in the next phase two loads a wave ask for the sub-tile two stages
// on that goes there.  A load has six to seven phases of eight to land; the wait is for a count
// (twelve younger loads a wave stay in flight, about 96 KB a CU), never for everything.
//
// A phase is two intervals between barriers: reading (LDS -> registers, the next loads) and
// multiplying.  The waves 4-7 run one interval behind the waves 0-3, and wave i and wave i + 4 share a
// SIMD: while one multiplies, the other reads, without either wave's code having to interleave the two.
//
// Measured with the chip's counters: 2,271 cycles a stage of 256 x 256 where the matrix instructions
// alone take 2,048 (90 %), whatever the caches hold.  With random operands on all CUs the chip then
// lowers its clock (2.4 -> 1.7 GHz): power bounds the large products now, not operands.
// Against the two-stage tiles before, in us: 2,048 x 28,672 x 4,096 (gate) 498 -> 369; 2,048 x 11,264 x
// 2,048 (gate) 104 -> 79; 2,048 x 6,144 x 4,096 99 -> 78; 2,048 x 4,096 x 14,336 212 -> 167; 500 x
// 22,016 x 4,096 (gate) 101 -> 79; 500 x 4,096 x 11,008 52 (8 slices) -> 43 (4); 1,500 x 5,632 x 2,048
// 49 -> 39; 72 x 2,048 x 2,048 11.2 -> 8.4.  Matrix instructions of 32 x 32 in place of 16 x 16 take 2,630
// cycles a stage (two chains of accumulators a phase do not cover their latency) at the same clock.
//
// float32 runs the same code on 16x16x4 instructions, four for the 16 bytes that a lane reads of either
// operand (which element of K a lane's operand stands for is free as long as A and B agree).  There
// the matrix unit's rate bounds everything, and what counts is that the CUs get equal numbers of tiles, three of
// 64 x 128 a CU at a time.  In us against the four-wave tiles of 128 x 128 before (and K in up to 16 slices for
// few rows): 700 x 11,264 x 2,048 with the gate 389 -> 264 (528 tiles of 128 x 128 on 256 CUs: three on some),
// 700 x 2,048 x 5,632 238 -> 141, 72 x 11,264 x 2,048 150 -> 76, 2,048 x 11,264 x 2,048 777 -> 697.  Tiles of
// 128 x 128 in this kernel: 900 x 11,264 x 2,048 510 (two a CU: what is left for the last round goes to
// CUs in pairs) against 384.
// A float32 sum's products go in two chains of accumulators, the halves of every phase's K, added at the
// end: a single one's rounding grows with the slice, and the slices are fewer than those of the tiles before (error
// against 64 bits, relative, with the four-wave tiles / one chain here / two: 65 x 2,048 x 5,632, in 16 / 8 / 8 slices, 3.4e-7 / 4.8e-7 /
// 3.4e-7; 1,500 x 2,560 x 2,048 5.7e-7 / 8.1e-7 / 5.7e-7; 700 x 5,632 x 2,048 with the gate 1.24e-6 / 1.24e-6 / 0.85e-6).
// It also leaves no product waiting for the one before it: 65 x 11,264 x 2,048 with the gate 80.2 -> 75.4 us, 700 rows
// 268 -> 264, 65 x 2,048 x 5,632 with the sum of its slices 33.3 -> 31.8, 1,500 x 4,096 x 4,096 386 -> 381.  Chains of 32 of
// K whose results are added in the loop leave less (1.8e-7 for 1,500 x 2,560 x 2,048) but cost 2 to 8 % more time.
// Three workgroups a CU leave 80 registers a wave, which the two chains just fit.
//
// The operands' roles are exchanged (A = W, B = X): a lane's four accumulators are four neighbouring
// columns of one row of Y, stored in one instruction.
#include "gemm_ring.hpp"

#include <math.h>

#include <type_traits>

#include "common.hpp"
#include "kllm_kernels.h"

namespace kllm {

__device__ __attribute__((aligned(16))) unsigned char g_ring_zeros[16];   // zero-initialised

// Neither the compiler's scheduler nor its memory operations cross this.
__device__ __forceinline__ void ring_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// This wave's LDS reads are done and at most VM of its loads are in flight.
template <int VM>
__device__ __forceinline__ void ring_wait() {
  static_assert(VM < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | ((VM >> 4) << 14) | 0x0070);
}

__device__ __forceinline__ void ring_barrier() {
  ring_fence();
  __builtin_amdgcn_s_barrier();
  ring_fence();
}

template <typename T> struct RingOperand;                // 16 bytes of a row
template <> struct RingOperand<bf16_t> { typedef bf16x8 type; };
template <> struct RingOperand<float> { typedef floatx4 type; };

template <bool WIDE> struct RingOffset { typedef unsigned type; };
template <> struct RingOffset<true> { typedef unsigned long type; };

__device__ __forceinline__ floatx4 ring_mma(bf16x8 a, bf16x8 b, floatx4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ floatx4 ring_mma(floatx4 a, floatx4 b, floatx4 acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
  return acc;
}

// WR x WC = 8 waves; a wave's part of a sub-tile of X is TM tiles of 16 rows, of W TN.  KIND of K: RING_WHOLE;
// RING_TAIL: some slice is no multiple of two stages, what lies behind its end is read as zeros; RING_LONG: also
// so long that a lane's offset from its tile's first row takes 64 bits.
enum : int { RING_WHOLE = 0, RING_TAIL = 1, RING_LONG = 2 };
constexpr int kRingLongK = 1 << 23;        // 255 rows of bfloat16, 127 of float32: below 2^32 bytes

template <typename T, typename TOUT, int MODE, int WR, int WC, int TM, int TN, int KIND>
__global__ __launch_bounds__(512, sizeof(T) == 4 ? 6 : 2) void gemm_ring_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                           TOUT* __restrict__ Y, int n, int m, int k, int tiles_x,
                                                           int tiles_y, int kslice, int act,
                                                           const float* __restrict__ act_params, int xcds, const RingRope rope) {
  constexpr bool ROPE = MODE == RING_ROPE, GATE = MODE == RING_GATE || ROPE, TAIL = KIND != RING_WHOLE;      // (GATE: columns in pairs)
  typedef typename RingOperand<T>::type op_t;
  typedef typename RingOffset<KIND == RING_LONG>::type off_t;
  constexpr int EPC = 16 / sizeof(T), STAGE = 8 * EPC;     // elements of a chunk of 16 bytes, of a stage
  constexpr int CHAINS = sizeof(T) == 4 ? 2 : 1;           // of products to a sum (see above)
  constexpr int XR = WR * TM * 16, WS = WC * TN * 16;      // rows of a sub-tile of X, of W
  constexpr int BM = 2 * XR, BN = GATE ? WS : 2 * WS;      // rows and columns of the output tile
  constexpr int XB = XR * 128, WB = WS * 128;              // bytes of a sub-tile
  static_assert(WR * WC == 8 && XR % 32 == 0 && WS % 32 == 0, "eight waves; whole or half load instructions");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];   // X [stage 2][half 2], then W likewise
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wr = wave / WC, wc = wave % WC, behind = wave / 4;

  // Workgroups are numbered so that the XCDs (which take them round-robin, each with an L2 of its own)
  // get contiguous runs of tiles, in bands of eight row tiles: a run covers about as many rows as columns.
  const int total = tiles_x * tiles_y;
  const int per_xcd = (total + xcds - 1) / xcds;
  const int id = ((int)blockIdx.x % xcds) * per_xcd + (int)blockIdx.x / xcds;
  if (id >= total) return;
  const int band = id / (8 * tiles_x), in_band = id - band * 8 * tiles_x;
  const int band_rows = min(8, tiles_y - band * 8);
  const int tcol = in_band / band_rows;
  const int row0 = (band * 8 + in_band - tcol * band_rows) * BM, col0 = tcol * BN;

  // blockIdx.y: a slice of K (a multiple of two stages, TAIL: of one); its sums go to Y[blockIdx.y]
  const int kbeg = blockIdx.y * kslice, klen = min(k, kbeg + kslice) - kbeg;    // (never empty)
  const int stages = TAIL ? (klen + 2 * STAGE - 1) / (2 * STAGE) * 2 : klen / STAGE;
  Y += (long)blockIdx.y * n * m;

  // Loads: a wave takes an eighth of a sub-tile's rows, eight rows an instruction (four, with half its
  // lanes, where it has only those left).  Lane l serves row l / 8 and, since such a load puts
  // its 16 bytes at LDS base + 16 l, slot l % 8 of that row.  Row r keeps chunk c (16 bytes) in slot
  // c ^ (r / 2 % 8), so that the 16-byte reads of 16 rows' chunk c meet all banks.  Rows that do not
  // exist are clamped to the last (their results are never stored).
  constexpr int XPW = XR / 8, WPW = WS / 8;                // rows per wave
  constexpr int XL = (XPW + 7) / 8, WL = (WPW + 7) / 8;    // load instructions per wave
  off_t xoff[2][XL], woff[2][WL];                        // bytes from the tile's first row, at K = kbeg
  int xchunk[XL], wchunk[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int r = XPW * wave + 8 * i + lane / 8;
    xchunk[i] = (lane % 8) ^ ((r >> 1) & 7);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      xoff[h][i] = (off_t)(min(row0 + h * XR + r, n - 1) - row0) * (off_t)k * (off_t)sizeof(T) + xchunk[i] * 16u;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int r = WPW * wave + 8 * i + lane / 8;
    wchunk[i] = (lane % 8) ^ ((r >> 1) & 7);
#pragma unroll
    for (int h = 0; h < 2; ++h)       // GATE: the first half of a tile's rows of W are gates, the second their up rows
      woff[h][i] = (off_t)(min(col0 + (GATE ? 0 : h * WS) + r, m - 1) - col0) * (off_t)k * (off_t)sizeof(T) + wchunk[i] * 16u;
    if constexpr (ROPE) {             // pair c is elements c % half and half + c % half of head c / half
      const int c = min(col0 + r, m - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) woff[h][i] = (off_t)(c + (c / rope.half + h) * rope.half) * (off_t)k * (off_t)sizeof(T) + wchunk[i] * 16u;
    }
  }
  const T* const xbase = X + (long)row0 * k + kbeg;
  const T* const wbase[2] = {W + (ROPE ? 0 : (long)col0 * k) + kbeg, W + (ROPE ? 0 : ((long)col0 + (GATE ? m : 0)) * k) + kbeg};

  auto load = [&](const char* src, off_t& off, int chunk, int left, unsigned char* dst) {
    if (CHAINS > 1) asm volatile("" : "+v"(off));        // (or the loop keeps 64-bit addresses instead: eight registers, spills)
    const char* at = src + off;
    if (TAIL) at = chunk * EPC < left ? at : reinterpret_cast<const char*>(g_ring_zeros);
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)at,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  };
  auto load_x = [&](int t, int h) {
    unsigned char* dst = lds + ((t & 1) * 2 + h) * XB + XPW * wave * 128;
    const char* src = reinterpret_cast<const char*>(xbase) + (long)t * 128;
#pragma unroll
    for (int i = 0; i < XL; ++i)
      if (XPW - 8 * i >= 8 || lane < 8 * (XPW - 8 * i)) load(src, xoff[h][i], xchunk[i], klen - STAGE * t, dst + 1024 * i);
  };
  auto load_w = [&](int t, int h) {
    unsigned char* dst = lds + 4 * XB + ((t & 1) * 2 + h) * WB + WPW * wave * 128;
    const char* src = reinterpret_cast<const char*>(wbase[h]) + (long)t * 128;
#pragma unroll
    for (int i = 0; i < WL; ++i)
      if (WPW - 8 * i >= 8 || lane < 8 * (WPW - 8 * i)) load(src, woff[h][i], wchunk[i], klen - STAGE * t, dst + 1024 * i);
  };

  // MFMA 16x16: lane l holds 16 bytes of row l % 16 of A from chunk l / 16 on, B likewise, D[4 (l / 16) + i][l % 16].
  const int lrow = lane % 16, lch = lane / 16;
  const int at = lrow * 128 + (lch ^ ((lrow >> 1) & 7)) * 16;       // (rows 16 apart share their permutation)
  const unsigned char* const xrd[2] = {lds + wr * TM * 2048 + at, lds + wr * TM * 2048 + (at ^ 64)};
  const unsigned char* const wrd[2] = {lds + 4 * XB + wc * TN * 2048 + at, lds + 4 * XB + wc * TN * 2048 + (at ^ 64)};
  op_t xf[TM][2], wf[2][TN][2];                           // [tile][half of the stage's K]
  auto read_x = [&](int parity, int h) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) xf[i][s] = *reinterpret_cast<const op_t*>(xrd[s] + (parity * 2 + h) * XB + i * 2048);
  };
  auto read_w = [&](int parity, int h) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s) wf[h][j][s] = *reinterpret_cast<const op_t*>(wrd[s] + (parity * 2 + h) * WB + j * 2048);
  };
  floatx4 acc[CHAINS][2][2][TM][TN];
#pragma unroll
  for (int s = 0; s < CHAINS; ++s)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[s][a][b][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int hx, int hw) {
    __builtin_amdgcn_s_setprio(1);                          // before the SIMD's other wave, which reads
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[s % CHAINS][hx][hw][i][j] = ring_mma(wf[hw][j][s], xf[i][s], acc[s % CHAINS][hx][hw][i][j]);
    __builtin_amdgcn_s_setprio(0);
  };

  // The order in which phases read the sub-tiles, one each: W0 | X0 W1 X1 W1' X0' W0' X1' W0'' | X0'' ...
  // (a dash: the next stage), and the loads are asked for in the same order.  A sub-tile is waited for in
  // the phase before the one that reads it, by every wave in front of that phase's first barrier: the
  // waves that run an interval behind have then waited before the others read.  Its buffer's last
  // readers have waited for their reads in front of that barrier too, a whole interval before the loads
  // that overwrite it are asked for.
  load_w(0, 0);
  load_x(0, 0);
  load_w(0, 1);
  load_x(0, 1);
  load_w(1, 1);
  load_x(1, 0);
  load_w(1, 0);
  load_x(1, 1);
  ring_fence();
  constexpr int KEEP = 3 * (XL + WL);                       // loads behind the sub-tile that the next phase reads
  ring_wait<KEEP>();
  ring_barrier();
  read_w(0, 0);
  ring_wait<KEEP>();
  ring_barrier();
  if (behind) ring_barrier();
#define KLLM_RING_PHASE(READ, LOAD, VM, HX, HW) \
  do {                                          \
    READ;                                       \
    LOAD;                                       \
    ring_fence();                               \
    ring_wait<(VM)>();                          \
    ring_barrier();                             \
    multiply(HX, HW);                           \
    ring_barrier();                             \
  } while (0)
  for (int t = 0; t + 2 < stages; t += 2) {
    KLLM_RING_PHASE(read_x(0, 0), load_w(t + 2, 0), KEEP, 0, 0);
    KLLM_RING_PHASE(read_w(0, 1), load_x(t + 2, 0), KEEP, 0, 1);
    KLLM_RING_PHASE(read_x(0, 1), load_w(t + 2, 1), KEEP, 1, 1);
    KLLM_RING_PHASE(read_w(1, 1), load_x(t + 2, 1), KEEP, 1, 0);
    KLLM_RING_PHASE(read_x(1, 0), load_w(t + 3, 1), KEEP, 0, 1);
    KLLM_RING_PHASE(read_w(1, 0), load_x(t + 3, 0), KEEP, 0, 0);
    KLLM_RING_PHASE(read_x(1, 1), load_w(t + 3, 0), KEEP, 1, 0);
    KLLM_RING_PHASE(read_w(0, 0), load_x(t + 3, 1), KEEP, 1, 1);
  }
  // the last two stages: nothing more is asked for, the waits count down what is still on its way
  KLLM_RING_PHASE(read_x(0, 0), , 3 * XL + 2 * WL, 0, 0);
  KLLM_RING_PHASE(read_w(0, 1), , 2 * XL + 2 * WL, 0, 1);
  KLLM_RING_PHASE(read_x(0, 1), , 2 * XL + WL, 1, 1);
  KLLM_RING_PHASE(read_w(1, 1), , XL + WL, 1, 0);
  KLLM_RING_PHASE(read_x(1, 0), , XL, 0, 1);
  KLLM_RING_PHASE(read_w(1, 0), , 0, 0, 0);
  KLLM_RING_PHASE(read_x(1, 1), , 0, 1, 0);
  multiply(1, 1);
  if (!behind) ring_barrier();
#undef KLLM_RING_PHASE

  float a_pos = 0.f, a_neg = 0.f;
  if (MODE == RING_UNARY && act == ACT_XIELU) {
    a_pos = softplus_f32(act_params[0]);
    a_neg = softplus_f32(act_params[1]);
  }
  auto sum = [&](int hx, int hw, int i, int j, int e) {
    return CHAINS == 1 ? acc[0][hx][hw][i][j][e] : acc[0][hx][hw][i][j][e] + acc[CHAINS - 1][hx][hw][i][j][e];
  };
  if constexpr (ROPE) {
    // A lane's four columns are four neighbouring pairs of a head.  The rows' pages are looked up where the tile has keys or values; a
    // value's place is beside its neighbour token's, so sixteen lanes fill a sector, as in rope_append.  In place of the 32-bit sums' way out and
    // back and rope_append's launch, in us: 2,048 x 2,560 x 2,048 33.0 + 9.0 and a gap -> 35.1; prompts of 2,048 at 1.1B Llama sizes 5,850 -> 5,720, of
    // 1,999 at 8B sizes 25,310 -> 24,850; 500 to 1,300 tokens, and 32-bit, the same to 0.3 %.
    typedef T tx4 __attribute__((ext_vector_type(4)));
    const int half = rope.half, hd = 2 * half, H = rope.H, KV = rope.KV, qd = H * hd, page_size = rope.page_size;
    const bool keys = rope.cache && col0 + WS > H * half;  // (a tile's columns may end behind the last pair)
    int head[TN], at[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int c = col0 + (wc * TN + j) * 16 + 4 * lch;
      head[j] = c / half;
      at[j] = c - head[j] * half;
      if (c >= m) head[j] = -1;
    }
    int page[2][TM] = {}, slot[2][TM] = {};
    if (keys) {
      int span[2][TM];
#pragma unroll
      for (int hx = 0; hx < 2; ++hx)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int r = min(row0 + hx * XR + (wr * TM + i) * 16 + lrow, n - 1);
          slot[hx][i] = rope.positions[r];
          span[hx][i] = rope.span_of_token[r];
        }
#pragma unroll
      for (int hx = 0; hx < 2; ++hx)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int p = slot[hx][i] / page_size;
          page[hx][i] = rope.block_table[(long)span[hx][i] * rope.max_pages + p];
          slot[hx][i] -= p * page_size;
        }
    }
    T* const cache = static_cast<T*>(rope.cache);
    const long block = (long)page_size * hd;
    // (the next row's turns are asked for while this one is stored; rows behind the last read that one's)
    floatx4 cs[2][TN], sn[2][TN];
    auto turn = [&](int t) {
      const int r = min(row0 + t / TM * XR + (wr * TM + t % TM) * 16 + lrow, n - 1);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        cs[t % 2][j] = floatx4{1.f, 1.f, 1.f, 1.f};
        sn[t % 2][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (rope.cos_t) {
          cs[t % 2][j] = *reinterpret_cast<const floatx4*>(rope.cos_t + (long)r * half + at[j]);
          sn[t % 2][j] = *reinterpret_cast<const floatx4*>(rope.sin_t + (long)r * half + at[j]);
        }
      }
    };
    turn(0);
#pragma unroll
    for (int t = 0; t < 2 * TM; ++t) {
      const int hx = t / TM, i = t % TM, r = row0 + hx * XR + (wr * TM + i) * 16 + lrow;
      if (t + 1 < 2 * TM) turn(t + 1);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        tx4 lo, hi;
        const bool value = head[j] >= H + KV;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = sum(hx, 0, i, j, e), b = sum(hx, 1, i, j, e);
          lo[e] = from_f32<T>(value ? a : a * cs[t % 2][j][e] - b * sn[t % 2][j][e]);
          hi[e] = from_f32<T>(value ? b : b * cs[t % 2][j][e] + a * sn[t % 2][j][e]);
        }
        if (r >= n || head[j] < 0) continue;
        if (!value) {
          T* o = head[j] < H ? Y + (long)r * qd + head[j] * hd
                             : cache + ((long)page[hx][i] * 2 * KV + head[j] - H) * block + (long)slot[hx][i] * hd;
          *reinterpret_cast<tx4*>(o + at[j]) = lo;
          *reinterpret_cast<tx4*>(o + at[j] + half) = hi;
        } else {
          T* v = cache + (((long)page[hx][i] * 2 + 1) * KV + head[j] - H - KV) * block + slot[hx][i];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[(long)(at[j] + e) * page_size] = lo[e];
            v[(long)(at[j] + e + half) * page_size] = hi[e];
          }
        }
      }
    }
    return;
  }
  const bool vec = m % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & (4 * sizeof(TOUT) - 1)) == 0;
  // KNOWN: the activation, where it has a copy of the stores of its own (-1: any).  Without a gate an activation went through the loop below (us, with that
  // and now: 1,500 x 5,632 x 2,048 with the squared rectifier 46.0 / 41.2, with SiLU 55.3 / 47.1, with GELU 57.8 / 46.1; 1,500 x 5,632 x 1,024 32.1 / 25.6,
  // 40.7 / 31.1 and 43.6 / 31.7).  For the gates one copy is as fast within 1 % (300 x 11,264 x 2,048 27.5 / 27.1, 700 37.7 / 37.5, 1,999 x 28,672 x
  // 4,096 374.8 / 375.1).
  auto store = [&](auto known) __attribute__((always_inline)) {
    constexpr int KNOWN = decltype(known)::value;
#pragma unroll
    for (int hx = 0; hx < 2; ++hx)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = row0 + hx * XR + (wr * TM + i) * 16 + lrow;
        if (r >= n) continue;
#pragma unroll
        for (int hw = 0; hw < (GATE ? 1 : 2); ++hw)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int c = col0 + hw * WS + (wc * TN + j) * 16 + 4 * lch;
            typedef TOUT vec_t __attribute__((ext_vector_type(4)));
            floatx4 q;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              q[e] = sum(hx, hw, i, j, e);
              if (GATE) q[e] = gate_act<TOUT>(q[e], KNOWN) * sum(hx, 1, i, j, e);
            }
            if constexpr (MODE == RING_UNARY) {
              // Larger tiles have one copy of the other activations to four sums: with four the kernel's end alone is longer than the
              // instruction cache, and at 256 x 256 its loops are no longer unrolled, so that the accumulators go through
              // scratch memory (tanh in us: 1,500 x 32,000 x 1,024 267 -> 162; 1,500 x 5,632 x 2,048
              // 68 -> 55; 700 x 5,632 x 2,048 49 -> 40).  Tiles of 128 x 128 are faster with four (300 x 2,048
              // x 2,048 24.2 / 28.5, with one 25.5 / 29.0).
              if constexpr (KNOWN < 0 && TM * TN >= 4) {
#pragma unroll 1
                for (int e = 0; e < 4; ++e) q = floatx4{q[1], q[2], q[3], unary_act<TOUT>(q[0], act, a_pos, a_neg)};
              } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) q[e] = unary_act<TOUT>(q[e], KNOWN < 0 ? act : KNOWN, a_pos, a_neg);
              }
            }
            vec_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = from_f32<TOUT>(q[e]);
            TOUT* dst = Y + (long)r * m + c;
            if (vec && c + 3 < m) {
              *reinterpret_cast<vec_t*>(dst) = v;
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (c + e < m) dst[e] = v[e];
            }
          }
      }
  };
  if constexpr (MODE == RING_GATE) {
    static_assert(ACT_COUNT == 2, "a copy of the stores for every gate");
    if (act == ACT_SILU) store(std::integral_constant<int, ACT_SILU>());
    else store(std::integral_constant<int, ACT_GELU_TANH>());
  } else if constexpr (MODE == RING_UNARY) {
    if (act == ACT_RELU_SQ) store(std::integral_constant<int, ACT_RELU_SQ>());
    else if (sizeof(TOUT) == 2 && act == ACT_GELU_TANH) store(std::integral_constant<int, ACT_GELU_TANH>());
    else if (sizeof(TOUT) == 2 && act == ACT_SILU) store(std::integral_constant<int, ACT_SILU>());
    else store(std::integral_constant<int, -1>());
  } else {
    store(std::integral_constant<int, -1>());
  }
}

// ------------------------------------------------------------------ which tile, how many slices of K
//
// Up to 64 rows of X (decode batches), where the weights' way from memory bounds the time, tiles of 64 rows:
// 64 x 128, three workgroups a CU, or in bfloat16 64 x 256, two a CU, where those are at most one a CU and
// the narrow ones more, with a slice of 512 of K at least (64 rows, in us, narrow / wide: 11,264 x 2,048 in 4
// slices 15.2 / 14.1; 12,288 x 4,096 in 4 24.5 / 22.3; in 8 24.6 / 27.8; 4,096 x 14,336 in 8 23.9 / 31.3;
// 2,560 x 2,048 in 16 8.1 / 9.3).  The two- and three-stage tiles of 64 x 64 and 64 x 128 before, at 64 rows: 11,264
// x 2,048 15.1, with the gate 30.3 (now 19.6); 12,288 x 4,096 28.4; 4,096 x 14,336 in 8 29.3; 28,672 x 4,096
// with the gate 61.2 (52.5); 2,048 x 2,048 in 8 6.4 (6.2); float32: 2,048 x 5,632 in 16 29.2 (in 16 slices of 352
// 20.8; in 15 of 384 19.2, in 11 22.9, in 8 28.9).
//
// More rows:
// A product's time in us is put together from what a tile costs a CU: rounds of the chip times (stages
// x a stage's time + what a tile costs beside its stages), against the time its weights need from
// memory, plus its output and a launch.  The constants for bfloat16 are fitted to a sweep of 13 numbers of rows
// from 72 to 2,048 and 12 sizes of W from 2,048 x 2,048 to 28,672 x 4,096, with every tile and 1 to 8
// slices (2,700 products on the full chip): the tile and slices that it chooses take 0.9 % longer than the fastest of
// the sweep on the mean, 12 % at worst.  It compares tiles, and is no forecast: single products of the sweep are 10 % around it
// (estimated / measured alone in us: 72 x 2,048 x 2,048 6.8 / 7.0; 1,500 x 2,048 x 5,632 40 / 41; 1,024 x 4,096 x 4,096 33 / 36), and
// where products run long enough for power to lower the clock every tile takes longer by about as much (2,048 x
// 28,672 x 4,096 with the gate 293 / 358 to 391 from run to run; 2,048 x 11,264 x 2,048 67 / 80 to 88; 500 x 22,016 x 4,096
// 64 / 72 to 79; 2,048 x 4,096 x 14,336 in two slices 136 / 163 to 175).  A 256 x 128 and a 128 x 192 tile were in the sweep too and won nothing
// that these four do not come within a per cent of.  float32: a stage's products at the rate that the
// matrix unit reaches (138 TFLOP/s on the chip); one workgroup alone on its CU took a third longer when the
// constants were made (a single chain of products a wave; two since).
struct RingTile {
  int rows, cols;          // of a product without a gate (with one: half as many columns)
  int per_cu;              // workgroups a CU holds
  float stage, tile;       // us a stage of 128 bytes of K (per_cu of them side by side), and beside the stages
  float stage_alone;       // ... with one workgroup on the CU
};
static const RingTile kRingTilesBf16[] = {
    {256, 256, 1, 1.04f, 3.0f, 1.04f}, {256, 192, 1, 0.835f, 2.6f, 0.835f}, {128, 256, 1, 0.68f, 1.4f, 0.68f},
    {128, 128, 2, 0.88f, 0.0f, 0.60f}};
constexpr int kRingNarrow = 4, kRingWide = 5;      // of up to 64 rows: 64 x 128, 64 x 256
static const RingTile kRingTilesF32[] = {{64, 128, 3, 2.94f, 1.0f, 1.30f}};
struct RingTiles {
  const RingTile* tile;
  int count, pair;         // elements of K in two stages
};
static RingTiles ring_tiles(bool f32) {
  if (f32) return {kRingTilesF32, 1, 64};
  return {kRingTilesBf16, 4, 128};
}

// K of a slice: whole pairs of stages; where that would leave the last slice empty, whole stages (the odd one's
// partner is read as zeros: as many stages as with pairs, but every workgroup has products).
static int ring_kslice(int k, int nsplit, int pair) {
  const int slice = ceil_div(ceil_div(k, nsplit), pair) * pair;
  return (long)slice * (nsplit - 1) < k ? slice : ceil_div(ceil_div(k, nsplit), pair / 2) * (pair / 2);
}

static float ring_time(const RingTile& t, int pair, int n, int m, int k, int nsplit, bool gate, int in_bytes, int out_bytes) {
  const long cus = device_cus();
  const long tiles = (long)ceil_div(n, t.rows) * ceil_div(m, gate ? t.cols / 2 : t.cols) * nsplit;
  const int stages = 2 * ceil_div(ring_kslice(k, nsplit, pair), pair);
  const long full = tiles / (t.per_cu * cus), rest = tiles % (t.per_cu * cus);
  float busy = (float)full * (stages * t.stage + t.tile);
  if (rest) {
    const int side = ceil_div(rest, cus);       // of them side by side on a CU
    busy += stages * (side == 1 ? t.stage_alone : t.stage * side / t.per_cu) + t.tile;
  }
  const float weights = 0.2e-6f * in_bytes * (gate ? 2.f : 1.f) * m * (float)k;      // 5 TB/s
  const float out = 0.2e-6f * out_bytes * nsplit * n * (float)m;
  const float b2 = busy * busy, w2 = weights * weights;
  return 3.3f + sqrtf(sqrtf(b2 * b2 + w2 * w2)) + out;
}

// (`us`: the estimate, written where there is one: not for k >= kRingLongK, nor for up to 64 rows of bfloat16.)
static int ring_tile(bool f32, int n, int m, int k, int nsplit, bool gate, bool f32_out, float* us = nullptr) {
  const RingTiles all = ring_tiles(f32);
  if (k >= kRingLongK) return f32 ? 0 : kRingNarrow;
  if (!f32 && n <= 64) {
    const long cus = device_cus(), narrow = (long)ceil_div(m, gate ? 64 : 128) * nsplit, wide = (long)ceil_div(m, gate ? 128 : 256) * nsplit;
    return narrow > cus && wide <= cus && ring_kslice(k, nsplit, all.pair) >= 512 ? kRingWide : kRingNarrow;
  }
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < all.count; ++i) {
    const float t = ring_time(all.tile[i], all.pair, n, m, k, nsplit, gate, f32 ? 4 : 2, f32_out ? 4 : 2);
    if (i == 0 || t < least) least = t, best = i;
  }
  if (us) *us = least;
  return best;
}

template <typename T, typename TOUT, int MODE, int WR, int WC, int TM, int TN, int KIND>
static int ring_launch(const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int act,
                       const float* act_params, const RingRope& rope, hipStream_t stream) {
  constexpr int XR = WR * TM * 16, WS = WC * TN * 16, BM = 2 * XR, BN = MODE == RING_GATE || MODE == RING_ROPE ? WS : 2 * WS;
  const int tx = ceil_div(m, BN), ty = ceil_div(n, BM), xcds = device_xcds();
  const dim3 grid(ceil_div((long)tx * ty, xcds) * xcds, nsplit);   // padded so that every XCD gets as many
  const size_t lds = (size_t)4 * (XR + WS) * 128;
  static int raised = 0;
  if (lds > 64 * 1024 && !raised) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_ring_kernel<T, TOUT, MODE, WR, WC, TM, TN, KIND>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) KLLM_FAIL((int)e, "gemm ring: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = 1;
  }
  hipLaunchKernelGGL((gemm_ring_kernel<T, TOUT, MODE, WR, WC, TM, TN, KIND>), grid, dim3(512), lds, stream, (const T*)x,
                     (const T*)w, (TOUT*)y, n, m, k, tx, ty, ring_kslice(k, nsplit, 256 / (int)sizeof(T)), act,
                     act_params, xcds, rope);
  return 0;
}

template <typename T, typename TOUT, int MODE, int KIND>
static int ring_shape(int tile, const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int act,
                      const float* ap, const RingRope& rope, hipStream_t st) {
  if constexpr (sizeof(T) == 2 && KIND != RING_LONG) {
    switch (tile) {
      case 0: return ring_launch<T, TOUT, MODE, 2, 4, 4, 2, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
      case 1: return ring_launch<T, TOUT, MODE, 4, 2, 2, 3, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
      case 2: return ring_launch<T, TOUT, MODE, 2, 4, 2, 2, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
      case 3: return ring_launch<T, TOUT, MODE, 2, 4, 2, 1, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
      case kRingWide: return ring_launch<T, TOUT, MODE, 2, 4, 1, 2, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
    }
  }
  return ring_launch<T, TOUT, MODE, 2, 4, 1, 1, KIND>(x, w, y, n, m, k, nsplit, act, ap, rope, st);
}

template <typename T, typename TOUT, int MODE>
static int ring_kind(int tile, const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int act,
                     const float* ap, const RingRope& rope, hipStream_t st) {
  constexpr int PAIR = 256 / sizeof(T);
  if constexpr (MODE != RING_ROPE)
    if (k >= kRingLongK) return ring_shape<T, TOUT, MODE, RING_LONG>(tile, x, w, y, n, m, k, nsplit, act, ap, rope, st);
  const int slice = ring_kslice(k, nsplit, PAIR);
  const bool whole = k % PAIR == 0 && slice % PAIR == 0;
  return whole ? ring_shape<T, TOUT, MODE, RING_WHOLE>(tile, x, w, y, n, m, k, nsplit, act, ap, rope, st)
               : ring_shape<T, TOUT, MODE, RING_TAIL>(tile, x, w, y, n, m, k, nsplit, act, ap, rope, st);
}

int gemm_ring(const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int mode, bool f32, bool f32_out,
              int act, const float* act_params, hipStream_t stream, const RingRope& rope) {
  const int tile = ring_tile(f32, n, m, k, nsplit, mode == RING_GATE || mode == RING_ROPE, f32_out);
  if (mode == RING_ROPE)
    return f32 ? ring_kind<float, float, RING_ROPE>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream)
               : ring_kind<bf16_t, bf16_t, RING_ROPE>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
  if (f32) {
    if (mode == RING_GATE) return ring_kind<float, float, RING_GATE>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
    if (mode == RING_UNARY) return ring_kind<float, float, RING_UNARY>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
    return ring_kind<float, float, RING_SUMS>(tile, x, w, y, n, m, k, nsplit, act, act_params, rope, stream);
  }
  if (mode == RING_GATE) return ring_kind<bf16_t, bf16_t, RING_GATE>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
  if (mode == RING_UNARY) return ring_kind<bf16_t, bf16_t, RING_UNARY>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
  if (f32_out) return ring_kind<bf16_t, float, RING_SUMS>(tile, x, w, y, n, m, k, nsplit, act, act_params, rope, stream);
  return ring_kind<bf16_t, bf16_t, RING_SUMS>(tile, x, w, y, n, m, k, 1, act, act_params, rope, stream);
}

}  // namespace kllm

using namespace kllm;

// The slices that take the least time together with the kernel that adds them: its reads beyond the
// 4.5 us that a launch takes whatever it holds (22 MB at 5 TB/s).  Slices of unequal length keep CUs
// waiting: cuts that leave more than a tenth of K unused are out.
// Where ring_tile does not estimate: one slice up to 64 rows of bfloat16 (decode batches, which their
// caller cuts by a rule of its own); eight, the most here, for a K so long that a lane's offset takes 64 bits:
// beside millions of products to a sum the slices' sums cost nothing.
extern "C" int kllm_gemm_prompt_slices(int n, int m, int k, int dtype) {
  if (n <= 0 || m <= 0 || k <= 0) return 1;
  const bool f32 = dtype == DT_F32;
  if (!f32 && n <= 64) return 1;
  if (k >= kRingLongK) return 8;
  int best = 1;
  float least = 0.f;
  for (int ns : {1, 2, 3, 4, 6, 8}) {
    const long pair = ring_tiles(f32).pair, slice = ceil_div(ceil_div(k, ns), (int)pair) * pair;
    if (ns > 1 && (slice * (ns - 1) >= k || 10 * slice * ns > 11L * k)) continue;
    float us = 0.f;
    ring_tile(f32, n, m, k, ns, false, true, &us);
    us += fmaxf(4.5f, 0.2e-6f * 4.f * ns * n * (float)m);
    if (ns == 1 || us < least) least = us, best = ns;
  }
  return best;
}

// Whether the product of n rows with the queries', keys' and values' weights goes to kllm_gemm_rope (all of K in one slice, rotated and
// appended in the product's end) or its slices to rope_append, which reads 4 bytes of each and writes 2 of every element.  Where the slices' estimate says
// one, the former always: the same product without its sums' way out and back.  Else where it is an eighth faster by the estimates, which leave out
// what the rotation costs the end of a tile (slices and append / one, us, and the estimates' share: 1,500 x 2,560 x 2,048 33.0 / 27.5, 0.82; 1,280
// rows 29.0 / 26.5, 0.86; left alone: 1,024 rows 26.0 / 25.7, 0.94; 1,024 x 6,144 x 4,096 59.5 / 62.7, 0.92; 450 x 12,288 x 4,096 63.9 / 63.3, 0.96).
extern "C" int kllm_gemm_rope_best(int n, int m, int k, int dtype) {
  if (n <= 64 || m <= 0 || k <= 0 || k >= kRingLongK) return 0;
  const int ns = kllm_gemm_prompt_slices(n, m, k, dtype);
  if (ns == 1) return 1;
  if (dtype == DT_F32) return 0;
  float one = 0.f, apart = 0.f;
  ring_tile(false, n, m / 2, k, 1, true, false, &one);
  ring_tile(false, n, m, k, ns, false, true, &apart);
  return one < 0.875f * (apart + fmaxf(4.5f, 0.2e-6f * (4 * ns + 2) * n * (float)m));
}

// Rows and columns of the tile that a product gets, as rows * 1000 + columns (of W's rows, gates included).
extern "C" int kllm_gemm_prompt_tile(int n, int m, int k, int nsplit, int gate, int dtype, int out_dtype) {
  if (n <= 0 || m <= 0 || k <= 0 || nsplit <= 0) return -1;
  const bool f32 = dtype == DT_F32;
  const int tile = ring_tile(f32, n, m, k, nsplit, gate != 0, out_dtype == DT_F32);
  if (!f32 && tile >= kRingNarrow) return 64000 + (tile == kRingWide ? 256 : 128);
  const RingTile& t = ring_tiles(f32).tile[tile];
  return t.rows * 1000 + t.cols;
}
