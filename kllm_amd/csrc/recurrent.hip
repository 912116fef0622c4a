// Recurrent mixers whose state is carried from token to token, and what they share.
//
// A short causal convolution per channel: y_t = sum_j w[c][j] x_(t - taps + 1 + j), zeros before
// position 0.  Its inputs of the last taps - 1 positions are part of a request's state: the
// kernels that convolve read them for the first tokens of a span, and a launch behind them (the scan, or
// `conv_state_update`) writes the span's last inputs there (one thread per request and channel reads the
// old entries before it writes the new ones).  In the scan's launch it costs 1.4 us (8 single tokens, 2,048 channels; 5 of a
// chain of 1,500 tokens) where a launch of its own takes 4.7, and the gap in front of it.
//
// The gated delta rule, per head with a state S [key channel][value channel]:
//
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
//
// with q and k unit vectors per head (q also times dk^-1/2), g = exp(-exp(A) softplus(a + dt))
// and beta = sigmoid(b).  `gated_delta_prep` turns the projections' sums into these (per token,
// parallel: convolution and SiLU of q, k, v, the unit norms, g, beta and the output gate),
// `gated_delta_scan` runs the recurrence (per request, head and block of value channels, token
// after token); the output's norm and gate are kllm_delta_out's.
//
// The gated linear recurrence, per channel: with u the convolved input, gates
// r = sigmoid(A_r u + b_r), i = sigmoid(A_i u + b_i) through block-diagonal matrices,
// log a = -c r (c = 8 softplus(lambda), prepared once), S <- a S + sqrt(1 - a^2) i u, and the
// output S * gelu(y) with y a second branch.  `linear_recurrence_prep` makes a and the added term
// for every token (parallel), `linear_recurrence_scan` runs the chain.
//
// States are 32-bit and start from zero where a span's first position is 0.  Everything here
// computes in 32-bit from the projections' 32-bit sums.
#include <math.h>

#include "common.hpp"
#include "conv.hpp"
#include "kllm_kernels.h"

namespace kllm {

constexpr int kRecThreads = 256;

__global__ __launch_bounds__(kRecThreads) void conv_state_update_kernel(
    const ConvTail tail, long slot_stride, const int* __restrict__ slots, const int* __restrict__ span_start,
    const int* __restrict__ span_pos) {
  const int c = blockIdx.x * kRecThreads + threadIdx.x;
  if (c >= tail.C) return;
  const int span = blockIdx.y;
  conv_tail(tail, slot_stride, c, slots[span], span_start[span], span_start[span + 1], span_pos[span] == 0);
}

// The same in the launch of a scan whose workgroups (span, head, block of columns) share the channels out.
__device__ __forceinline__ void conv_tail_of_span(const ConvTail& tail, long slot_stride, int slot, long t0, long t1,
                                                  bool fresh) {
  const int threads = gridDim.y * gridDim.z * kRecThreads;
  for (int c = (blockIdx.y * gridDim.z + blockIdx.z) * kRecThreads + threadIdx.x; tail.taps > 1 && c < tail.C; c += threads)
    conv_tail(tail, slot_stride, c, slot, t0, t1, fresh);
}

// ---------------------------------------------------------------------------- gated delta rule

// proj: [nsplit][n][cols], columns q (G*dk) | k (G*dk) | v (H*dv) | b (H) | a (H) | gate (H*dv) |
// whatever else the product made.  With `a_sums` ([a_ns][n][a_row], the first H*dk of a row) the
// decay has one number per head and key channel, from sums of their own, and proj has no a
// columns; with `gate_sums` ([g_ns][n][g_row], the first H*dv of a row) the gate's sums are their
// own too and proj has no gate columns.
// One wave per (token, item): the items are the G query heads, the G key heads and the H value
// heads; a value head's wave also makes that head's gate, decays and beta.  A lane keeps up to
// four channels of a query or key head (heads of up to 256) between the sum and the division.
//
// Bound by a decode batch's trips to memory in a row and, for a prompt, by the sums' bytes: with four taps a wave asks for its channels' rows,
// weights and, where the span begins inside the window, entries at once, 128 channels at a time (tap after tap waited for each; 8 tokens, heads of 128: 8.6 -> 6.9 us, 1,500 tokens 55.7 -> 33.4).
// TAPS: their number up to four, 0 for more, which go a channel and a tap at a time.  R: channels a lane takes at a time, of heads up to 64 one.  us, 1,500 tokens:
// three taps, 16 heads of 64, tap after tap 17.3, and of 128 channels at a time, the head's or not, 22.5, so 13.2; 32 heads of 128 46.6, so 27.9; four
// taps, 16 heads of 64, tap after tap 20.9, two channels a lane 15.2, one 14.7.
template <int TAPS, int R>
__global__ __launch_bounds__(kRecThreads) void gated_delta_prep_kernel(
    const int* __restrict__ span_of_token, const int* __restrict__ span_start, const int* __restrict__ span_pos, const int* __restrict__ slots,
    const float* __restrict__ proj, int H, int G, int dk, int dv, const float* __restrict__ conv_w, int taps, int nsplit, long cols, long split_stride,
    const float* __restrict__ state, long slot_stride, const float* __restrict__ a_log, const float* __restrict__ dt_bias, float* __restrict__ qn,
    float* __restrict__ kn, float* __restrict__ vv, float* __restrict__ gb, float* __restrict__ gate, float unit_eps,
    const float* __restrict__ a_sums, int a_ns, long a_stride, long a_row,
    const float* __restrict__ gate_sums, int g_ns, long g_stride, long g_row, int gate_sigmoid,
    float* __restrict__ dec) {
  const long t = blockIdx.x;
  int at = blockIdx.x;                                   // (vector loads: scalar ones come one behind the other)
  asm volatile("" : "+v"(at));
  const int span_v = span_of_token[at];
  asm volatile("" ::"s"(conv_w), "s"(taps), "s"(nsplit), "s"(cols), "s"(split_stride), "s"(state), "s"(slot_stride), "s"(a_log), "s"(dt_bias), "s"(qn),
               "s"(kn), "s"(vv), "s"(gb), "s"(gate), "s"(unit_eps), "s"(a_sums), "s"(gate_sums));
  const int first_v = span_start[span_v], pos_v = span_pos[span_v], slot_v = slots[span_v];
  const int lane = threadIdx.x % kWave;
  const int item = blockIdx.y * (kRecThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (item >= 2 * G + H) return;
  const int QK = G * dk, HV = H * dv, C = 2 * QK + HV, K = TAPS ? TAPS - 1 : taps - 1;
  constexpr int FROM = 4 - TAPS;                         // of four rows up to the token's, the first that the convolution has (TAPS)
  const int gate_col = C + (a_sums ? H : 2 * H);
  // y[r]: SiLU of the convolution of channel c0 + lane + 64 r, of `width` (beyond it some channel's, not used)
  struct Ask {                                           // what four taps need, on its way
    float x[R][4], w[R][4];
  };
  auto ask = [&](int c0, int width, int e0) -> Ask {
    Ask A;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int c = c0 + min(e0 + lane + kWave * r, width - 1);
#pragma unroll
      for (int j = FROM; j < 4; ++j) {                   // (rows that are not there: the step's first, not used)
        A.x[r][j] = proj[max(t - 3 + j, 0L) * cols + c];
        A.w[r][j] = conv_w[(long)c * TAPS + j - FROM];
      }
    }
    return A;
  };
  auto convolved = [&](Ask& A, int c0, int width, int e0, float (&y)[R]) {
    const long t0 = __builtin_amdgcn_readfirstlane(first_v);
    const bool fresh = __builtin_amdgcn_readfirstlane(pos_v) == 0;
    const float* st = state + (long)__builtin_amdgcn_readfirstlane(slot_v) * slot_stride;
    if constexpr (TAPS > 0) {
      const int before = (int)min(max(t0 - t + 3, 0L), 3L);      // rows of the window before the span's first: entries of the state, the last K of three
      float was[R][3];
      if (before > 0 && !fresh) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = FROM; j < 3; ++j) was[r][j] = st[(long)(c0 + min(e0 + lane + kWave * r, width - 1)) * K + j - FROM];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        y[r] = 0.f;
        const int c = c0 + min(e0 + lane + kWave * r, width - 1);
        for (int s = 1; s < nsplit; ++s)
#pragma unroll
          for (int j = FROM; j < 4; ++j) A.x[r][j] += proj[s * split_stride + max(t - 3 + j, 0L) * cols + c];
#pragma unroll
        for (int j = FROM; j < 4; ++j) {
          float in = A.x[r][j];
          if (j < before) {                              // row t - 3 + j, before - j rows before the first: entry K - (before - j)
            in = 0.f;
            if (!fresh) in = before - j == 1 ? was[r][2] : before - j == 2 ? was[r][1] : was[r][0];
          }
          y[r] = fmaf(A.w[r][j], in, y[r]);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int c = c0 + e0 + lane + kWave * r;
        y[r] = 0.f;
        if (c < c0 + width)
          y[r] = conv_at(proj, nsplit, split_stride, cols, c, nullptr, conv_w + (long)c * taps, taps, st + (long)c * K, fresh, t, t0);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] /= 1.f + expf(-y[r]);       // SiLU
  };
  if (item < 2 * G) {        // a head of q or k: the unit norm
    const int c0 = item * dk;                            // q's heads, then k's, lie side by side
    float val[4] = {0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
#pragma unroll
    for (int h = 0; h < 4 / R; ++h) {
      if (h * R * kWave >= dk) break;
      float y[R];
      Ask A;
      if (TAPS) A = ask(c0, dk, h * R * kWave);
      convolved(A, c0, dk, h * R * kWave, y);
#pragma unroll
      for (int r = 0; r < R; ++r) val[R * h + r] = lane + kWave * (R * h + r) < dk ? y[r] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) ss = fmaf(val[r], val[r], ss);
    ss = wave_sum(ss);
    const bool is_q = item < G;
    const float f = (is_q ? 1.f / sqrtf((float)dk) : 1.f) / sqrtf(ss + unit_eps);
    float* dst = is_q ? qn + t * QK + (long)item * dk : kn + t * QK + (long)(item - G) * dk;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = lane + kWave * r;
      if (e < dk) dst[e] = val[r] * f;
    }
    return;
  }
  const int h = item - 2 * G;
  // the head's decay and beta: what they are made of is asked for first
  const bool own_decay = !a_sums;
  float pb = proj[t * cols + C + h], pa = proj[t * cols + C + (own_decay ? H + h : h)];
  const float al = a_log[h], dt = dt_bias[own_decay ? h : 0];
  for (int e0 = 0; e0 < dv; e0 += R * kWave) {
    Ask A;
    if (TAPS) A = ask(2 * QK + h * dv, dv, e0);
    float g[R], y[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int c = h * dv + min(e0 + lane + kWave * r, dv - 1);
      const float* from = gate_sums ? gate_sums + t * g_row + c : proj + t * cols + gate_col + c;
      g[r] = from[0];
    }
    for (int s = 1; s < (gate_sums ? g_ns : nsplit); ++s)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int c = h * dv + min(e0 + lane + kWave * r, dv - 1);
        g[r] += gate_sums ? gate_sums[s * g_stride + t * g_row + c] : proj[s * split_stride + t * cols + gate_col + c];
      }
    convolved(A, 2 * QK + h * dv, dv, e0, y);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = e0 + lane + kWave * r;
      if (e >= dv) break;
      vv[t * HV + h * dv + e] = y[r];
      gate[t * HV + h * dv + e] = gate_sigmoid ? sigmoid_f32(g[r]) : g[r] / (1.f + expf(-g[r]));
    }
  }
  if (a_sums) {       // one decay per head and key channel; dt_bias has as many entries
    const float rate = expf(al);
    for (int e = lane; e < dk; e += kWave) {
      const int c = h * dk + e;
      float a = 0.f;
      for (int s = 0; s < a_ns; ++s) a += a_sums[s * a_stride + t * a_row + c];
      dec[t * (long)H * dk + c] = expf(-rate * softplus_f32(a + dt_bias[c]));
    }
  }
  if (lane == 0) {
    for (int s = 1; s < nsplit; ++s) {
      pb += proj[s * split_stride + t * cols + C + h];
      if (own_decay) pa += proj[s * split_stride + t * cols + C + H + h];
    }
    gb[t * 2 * H + h] = own_decay ? expf(-expf(al) * softplus_f32(pa + dt)) : 1.f;
    gb[t * 2 * H + H + h] = sigmoid_f32(pb);
  }
}

constexpr int kDeltaParts = 16;                              // lanes that share a column of the state
constexpr int kDeltaCols = kRecThreads / kDeltaParts;        // columns of a workgroup
constexpr int kDeltaBlock = 16;                              // tokens staged at a time

// Thread (j, p): column j of the workgroup's block of value channels, and of the state's rows the
// runs of four that begin at 4 p, 64 + 4 p, ...: NB runs.  A block of tokens' vectors goes through
// LDS, rows padded with zeros to 64 NB: k and q, v [16 columns], and {g, beta, k . q} per token; the
// sums over a column's rows are lane exchanges within its sixteen lanes.
// What bounds it is the chain from token to token on one wave a SIMD.  With D S the decayed state,
//   u = beta (v - (D S)^T k),   S' = D S + k u^T,   o = S'^T q = (D S)^T q + (k . q) u,
// so that both sums over the rows are made of the same numbers, run side by side and neither waits
// for u; k . q comes from the staging.  Rows lie so that a lane reads four with one 16-byte LDS read
// (sixteen reads of 4 bytes a token before), the next token's while this one is computed.
// 1,500 tokens, 16 heads of 128 x 128: 635 -> 263 us.
// VEC: the decay has one number per head and key channel (`dec` [n][H*dk], staged like the keys)
// instead of one per head.
template <int NB, bool VEC>
__global__ __launch_bounds__(kRecThreads) void gated_delta_scan_kernel(
    const int* __restrict__ span_start, const int* __restrict__ slots, const int* __restrict__ span_pos, float* __restrict__ state, int H, int G,
    int dk, int dv, long slot_stride, const float* __restrict__ kn, const float* __restrict__ qn, const float* __restrict__ vv,
    const float* __restrict__ gb, float* __restrict__ o_out, const float* __restrict__ dec, const ConvTail tail) {
  constexpr int ROW = 64 * NB;                       // a token's row in LDS
  constexpr int NV = VEC ? 3 : 2;                    // vectors of a token: k, q and the decays
  __shared__ __attribute__((aligned(16))) float rows[NV][kDeltaBlock][ROW];
  __shared__ float vs[kDeltaBlock][kDeltaCols], os[kDeltaBlock][kDeltaCols];
  __shared__ __attribute__((aligned(16))) float gs[kDeltaBlock][4];      // g, beta, k . q
  int at = blockIdx.x;                               // (vector loads: scalar ones come one behind the other)
  asm volatile("" : "+v"(at));
  const int first_v = span_start[at], last_v = span_start[at + 1], slot_v = slots[at], pos_v = span_pos[at];
  asm volatile("" ::"s"(kn), "s"(qn), "s"(vv), "s"(gb), "s"(o_out), "s"(dec), "s"(tail.proj), "s"(tail.split_stride), "s"(tail.cols), "s"(tail.in_bias),
               "s"(tail.state), "s"(tail.nsplit), "s"(tail.col0), "s"(tail.C), "s"(tail.taps));
  const int h = blockIdx.y, tid = threadIdx.x;
  const int g = h / (H / G);
  const int jl = tid / kDeltaParts, p = tid % kDeltaParts;
  const int j = blockIdx.z * kDeltaCols + jl;
  const bool col = j < dv;
  const long t0 = __builtin_amdgcn_readfirstlane(first_v), t1 = __builtin_amdgcn_readfirstlane(last_v);
  const int slot = __builtin_amdgcn_readfirstlane(slot_v);
  const bool fresh = __builtin_amdgcn_readfirstlane(pos_v) == 0;
  float* S = state + (long)slot * slot_stride + (long)h * dk * dv;
  if (t1 - t0 == 1 && dv % 4 == 0 && (((unsigned long)S | (unsigned long)vv) & 15) == 0) {
    // One token: the state's way from memory and back is all there is.  A thread takes four columns of every 64th row, 16 bytes a load,
    // and the sums over the rows go over the wave's sixteen rows by lane exchanges and over the waves through LDS.  8 tokens, 16 heads of
    // 128 x 128: 13.3 -> 7.2 us (17 MB; 16-byte pieces of four rows a load before, and a chain's staging for one token).
    const int quad = tid % 4, rr = tid / 4;
    const int j4 = blockIdx.z * kDeltaCols + 4 * quad, jc = j4 < dv ? j4 : 0;
    const long key = t0 * G * dk + (long)g * dk, head = t0 * H + h;
    floatx4 x[NB];
    float k[NB], q[NB], d[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int r = min(64 * b + rr, dk - 1);
      k[b] = kn[key + r];
      q[b] = qn[key + r];
      d[b] = VEC ? dec[head * dk + r] : 1.f;
    }
    const float decay = gb[2 * t0 * H + h], beta = gb[2 * t0 * H + H + h];
    const floatx4 v = *reinterpret_cast<const floatx4*>(vv + head * dv + jc);
#pragma unroll
    for (int b = 0; b < NB; ++b) x[b] = *reinterpret_cast<const floatx4*>(S + (long)min(64 * b + rr, dk - 1) * dv + jc);
    conv_tail_of_span(tail, slot_stride, slot, t0, t1, fresh);
    float kq = 0.f, dks[4] = {0.f, 0.f, 0.f, 0.f}, dqs[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const bool row = 64 * b + rr < dk;
      k[b] = row ? k[b] : 0.f;
      q[b] = row ? q[b] : 0.f;
      kq = fmaf(k[b], q[b], kq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[b][e] = row && !fresh ? x[b][e] * (VEC ? d[b] : decay) : 0.f;
        dks[e] = fmaf(x[b][e], k[b], dks[e]);
        dqs[e] = fmaf(x[b][e], q[b], dqs[e]);
      }
    }
    auto over_rows = [](float v) { return group4_sum(dpp_add<0x128>(dpp_add<0x124>(v))); };      // row_ror 4 and 8: lanes of the same quad
    floatx4(*meet)[4][4] = reinterpret_cast<floatx4(*)[4][4]>(&rows[0][0][0]);      // [wave][quad]: k . S, q . S, k . q
    floatx4 dk4, dq4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dk4[e] = over_rows(dks[e]);
      dq4[e] = over_rows(dqs[e]);
    }
    kq = over_rows(kq);
    if (tid % kWave < 4) {
      meet[tid / kWave][quad][0] = dk4;
      meet[tid / kWave][quad][1] = dq4;
      meet[tid / kWave][quad][2][0] = kq;
    }
    __syncthreads();
    dk4 = meet[0][quad][0];
    dq4 = meet[0][quad][1];
    kq = meet[0][quad][2][0];
#pragma unroll
    for (int w = 1; w < kRecThreads / kWave; ++w) {
      dk4 += meet[w][quad][0];
      dq4 += meet[w][quad][1];
      kq += meet[w][quad][2][0];
    }
    const floatx4 u = beta * (v - dk4);
    if (j4 >= dv) return;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (64 * b + rr >= dk) break;
      floatx4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fmaf(k[b], u[e], x[b][e]);
      *reinterpret_cast<floatx4*>(S + (long)(64 * b + rr) * dv + j4) = y;
    }
    if (tid < 4)
#pragma unroll
      for (int e = 0; e < 4; ++e) o_out[head * dv + j4 + e] = fmaf(kq, u[e], dq4[e]);
    return;
  }
  floatx4 s[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 64 * b + 4 * p + e;
      s[b][e] = (col && r < dk && !fresh) ? S[(long)r * dv + j] : 0.f;
    }
  conv_tail_of_span(tail, slot_stride, slot, t0, t1, fresh);
  const int QK = G * dk, HV = H * dv;
  // A thread's pieces of a block of tokens: of each vector the elements tid % 64 + 64 i of tokens
  // tid / 64 + 4 q, one of v, one of g and beta.  They are asked for one block ahead and wait in
  // registers while the block before them is multiplied.  A token that is not there decays nothing
  // and writes nothing: k = q = 0, g = 1, beta = 0.
  const int e0 = tid % 64, r0 = tid / 64;
  const int v_tt = tid / kDeltaCols, v_c = blockIdx.z * kDeltaCols + tid % kDeltaCols;
  struct Pieces {
    float x[NV][4][NB], v, g;
  };
  auto fetch = [&](long tb, int nt) -> Pieces {
    Pieces P;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int tt = r0 + 4 * q, e = e0 + 64 * i;
        const bool ok = tt < nt && e < dk;
        const long at = (tb + (ok ? tt : 0)) * QK + (long)g * dk + (ok ? e : 0);
        P.x[0][q][i] = ok ? kn[at] : 0.f;
        P.x[1][q][i] = ok ? qn[at] : 0.f;
        if constexpr (VEC) P.x[2][q][i] = ok ? dec[(tb + tt) * (long)H * dk + (long)h * dk + e] : 1.f;
      }
    P.v = (v_tt < nt && v_c < dv) ? vv[(tb + v_tt) * HV + (long)h * dv + v_c] : 0.f;
    P.g = tid < 2 * nt ? gb[(tb + tid / 2) * 2 * H + (tid % 2) * H + h] : tid % 2 ? 0.f : 1.f;
    return P;
  };
  long tb = t0;
  int nt = (int)min((long)kDeltaBlock, t1 - tb);
  Pieces pre = fetch(tb, nt);
  while (tb < t1) {
    __syncthreads();                                 // the block before this one has been read
#pragma unroll
    for (int x = 0; x < NV; ++x)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < NB; ++i) rows[x][r0 + 4 * q][e0 + 64 * i] = pre.x[x][q][i];
    vs[v_tt][tid % kDeltaCols] = pre.v;
    if (tid < 2 * kDeltaBlock) gs[tid / 2][tid % 2] = pre.g;
    __syncthreads();
    const long tb_next = tb + kDeltaBlock;
    const int nt_next = (int)max(0L, min((long)kDeltaBlock, t1 - tb_next));
    if (nt_next > 0) pre = fetch(tb_next, nt_next);
    {   // k . q: sixteen lanes a token
      float kq = 0.f;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const floatx4 kv = *reinterpret_cast<const floatx4*>(&rows[0][jl][64 * b + 4 * p]);
        const floatx4 qv = *reinterpret_cast<const floatx4*>(&rows[1][jl][64 * b + 4 * p]);
#pragma unroll
        for (int e = 0; e < 4; ++e) kq = fmaf(kv[e], qv[e], kq);
      }
      kq = parts_sum<kDeltaParts>(kq);
      if (p == 0) gs[jl][2] = kq;
    }
    __syncthreads();
    struct Token {
      floatx4 k[NB], q[NB], d[VEC ? NB : 1], g;
      float v;
    };
    auto read = [&](int tt, Token& T) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        T.k[b] = *reinterpret_cast<const floatx4*>(&rows[0][tt][64 * b + 4 * p]);
        T.q[b] = *reinterpret_cast<const floatx4*>(&rows[1][tt][64 * b + 4 * p]);
        if constexpr (VEC) T.d[b] = *reinterpret_cast<const floatx4*>(&rows[NV - 1][tt][64 * b + 4 * p]);
      }
      T.g = *reinterpret_cast<const floatx4*>(&gs[tt][0]);
      T.v = vs[tt][jl];
    };
    float kept = 0.f;                                // token p's output of this column
    Token T[2];
    read(0, T[0]);
    for (int t4 = 0; t4 < nt; t4 += 4) {             // (tokens behind the last change nothing)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tt = t4 + i;
        read(min(tt + 1, kDeltaBlock - 1), T[(i + 1) & 1]);
        const Token& C = T[i & 1];
        float dk0 = 0.f, dk1 = 0.f, dq0 = 0.f, dq1 = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (VEC) s[b][e] *= C.d[b][e]; else s[b][e] *= C.g[0];
            float& a = e & 1 ? dk1 : dk0;
            float& c = e & 1 ? dq1 : dq0;
            a = fmaf(s[b][e], C.k[b][e], a);
            c = fmaf(s[b][e], C.q[b][e], c);
          }
        const float dot = parts_sum<kDeltaParts>(dk0 + dk1), dq = parts_sum<kDeltaParts>(dq0 + dq1);
        const float u = tt < nt ? C.g[1] * (C.v - dot) : 0.f;      // (0 also where the state is not finite)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[b][e] = fmaf(C.k[b][e], u, s[b][e]);
        const float o = fmaf(C.g[2], u, dq);
        kept = p == tt ? o : kept;
      }
    }
    os[p][jl] = kept;
    __syncthreads();
    if (v_tt < nt && v_c < dv) o_out[(tb + v_tt) * HV + (long)h * dv + v_c] = os[v_tt][tid % kDeltaCols];
    tb = tb_next;
    nt = nt_next;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 64 * b + 4 * p + e;
      if (col && r < dk) S[(long)r * dv + j] = s[b][e];
    }
}

// The same recurrence with one decay a head, sixteen tokens of a span at a time.  From the state S in front of them,
// with G_i the product of the decays up to token i and G_ij that of those behind token j up to i,
//   x_i = v_i - G_i (S^T k_i)          u_i = beta_i (x_i - sum_(j<i) G_ij (k_j . k_i) u_j)
//   o_i = G_i (S^T q_i) + sum_(j<=i) G_ij (k_j . q_i) u_j          S' = G_15 S + sum_i G_15,i k_i u_i^T
// u = M x with M = (1 + L)^-1 diag(beta), L_ij = beta_i G_ij (k_j . k_i) below the diagonal: what does not hang on the state
// is made for all sixteens at once (`gated_delta_factors`), and the chain of a sixteen is matrix products.
// Token by token each wave reads every token's key and query out of LDS and waits for two sums over its lanes; here
// a sixteen takes 2,070 cycles, of which 928 are matrix instructions.  In us, token by token and both kernels here (the
// factors' share), 16 heads of 128 x 128: 1,500 tokens 269 / 98 (12), 8 x 256 109 / 65 (14), 480 beside 8 single tokens 118 / 61 (9),
// 64 16.6 / 13.3 (6).  Relative errors of the outputs against 64 bits, weak to strong decays: 1.9e-7 / 1.3e-7, 9.6e-8 / 8.6e-8,
// 8.8e-8 / 7.1e-8.  Measured and not taken: four tokens at a time by 4 x 4 matrix instructions (236), sums of the waves'
// shares in an order of each wave's own, the update's products before the outputs' (104).
constexpr int kSixteen = 16;
// The factors of a sixteen, in the order that the scan's lanes read them (tokens that are not there: zeros, decays of one).
// Per head of keys: keys [channel / 4][token][4], queries likewise, keys [token / 4][channel][4]; channels in multiples of 64.
// Per head: M [token j / 4][token i][4], G_ij (k_j . q_i) [j % 4][j / 4][i], (G_i, G_15,i) [i].
// The sixteens of span s begin at number t0 / 16 + s of all (each span has one more than its sixteenth of the tokens at most).
constexpr int kHeadFactors = 2 * kSixteen * kSixteen + 2 * kSixteen;

__host__ __device__ inline long sixteen_floats(int H, int G, int rows) {
  return (long)G * 3 * kSixteen * rows + (long)H * kHeadFactors;
}

typedef double doublex4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ float dpp_moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Four lanes' four numbers: lane l's number e becomes lane e's number l.
__device__ __forceinline__ void transpose_four(floatx4& x, int lane) {
  const bool odd = lane & 1, high = lane & 2;
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    const float got = dpp_moved<0xB1>(odd ? x[e] : x[e + 1]);
    x[e] = odd ? got : x[e];
    x[e + 1] = odd ? x[e + 1] : got;
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float got = dpp_moved<0x4E>(high ? x[e] : x[e + 2]);
    x[e] = high ? got : x[e];
    x[e + 2] = high ? x[e + 2] : got;
  }
}

// Workgroup (sixteen, head of keys).  The sums go by the 64-bit matrix instruction (wave w takes the channels 16 w + 64 i),
// then a wave makes a head's factors.  L to the power of 16 is zero, so that (1 + L)^-1 = (1 + L^8) (1 + L^4) (1 + L^2)
// (1 - L); an operand on the left is read from its transpose in the layout of a result, so every power is made with
// its transpose.  Everything is 64-bit until it is written.
template <int NB, bool V4>
__global__ __launch_bounds__(kRecThreads, NB <= 2 && V4 ? 4 : 2) void gated_delta_factors_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn, const float* __restrict__ gb,
    const int* __restrict__ span_start, float* __restrict__ factors, int n_spans, int H, int G, int dk) {
  constexpr int T = kSixteen, WAVES = kRecThreads / kWave, ROWS = 64 * NB;
  __shared__ doublex4 part[2][WAVES][kWave];
  __shared__ double runs[WAVES][4][T];               // runs[w][p][l]: the decays of the 2^p tokens up to l
  const int g = blockIdx.y, per = H / G, lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), low = lane % 16, high = lane / 16;
  const int QK = G * dk;
  auto mul = [](const doublex4& left_t, const doublex4& right, doublex4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f64_16x16x4f64(left_t[e], right[e], c, 0, 0, 0);
    return c;
  };
  const int number = blockIdx.x;
  int span = -1;                                     // the last span that begins at this sixteen or before it
  for (int s0 = 0; s0 < n_spans; s0 += kWave) {
    const int s = min(s0 + lane, n_spans - 1);
    const unsigned long long at = __ballot(s0 + lane < n_spans && span_start[s] / T + s <= number);
    span += __popcll(at);
    if (at != ~0ull) break;
  }
  const int t0 = span_start[span], t1 = span_start[span + 1];
  const int t = t0 + (number - t0 / T - span) * T;
  if (t >= t1) return;
  const int nt = min(T, t1 - t), tok = t + min(low, nt - 1);
  const bool there = low < nt;
  const float* krow = kn + (long)tok * QK + (long)g * dk;
  const float* qrow = qn + (long)tok * QK + (long)g * dk;
  const float* grow = gb + (long)tok * 2 * H + g * per + min(wave, per - 1);
  floatx4 k[NB], q[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int r = 16 * wave + 64 * c + 4 * high;
    if constexpr (V4) {
      k[c] = *reinterpret_cast<const floatx4*>(krow + min(r, dk - 4));
      q[c] = *reinterpret_cast<const floatx4*>(qrow + min(r, dk - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k[c][e] = krow[min(r + e, dk - 1)];
        q[c][e] = qrow[min(r + e, dk - 1)];
      }
    }
  }
  float d_low = grow[0], b_low = grow[H];
  doublex4 kk = {0., 0., 0., 0.}, qk = {0., 0., 0., 0.};
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool ok = there && 16 * wave + 64 * c + 4 * high + e < dk;
      k[c][e] = ok ? k[c][e] : 0.f;
      q[c][e] = ok ? q[c][e] : 0.f;
      const double kd = k[c][e], qd = q[c][e];
      kk = __builtin_amdgcn_mfma_f64_16x16x4f64(kd, kd, kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f64_16x16x4f64(qd, kd, qk, 0, 0, 0);
    }
  float* of_sixteen = factors + number * sixteen_floats(H, G, ROWS);
  float* keys = of_sixteen + (long)g * 3 * T * ROWS;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int quad = 4 * wave + 16 * c + high;
    *reinterpret_cast<floatx4*>(keys + (quad * T + low) * 4) = k[c];
    *reinterpret_cast<floatx4*>(keys + T * ROWS + (quad * T + low) * 4) = q[c];
    transpose_four(k[c], lane);                    // tokens low / 4 * 4 .. + 3 of channel 4 quad + low % 4
    *reinterpret_cast<floatx4*>(keys + 2 * T * ROWS + (low / 4 * ROWS + 4 * quad + low % 4) * 4) = k[c];
  }
  part[0][wave][lane] = kk;                        // element e of a result: row 4 e + high, column low
  part[1][wave][lane] = qk;
  __syncthreads();
  for (int hh = wave; hh < per; hh += WAVES) {
    const int h = g * per + hh;
    if (hh > wave) {
      d_low = gb[(long)tok * 2 * H + h];
      b_low = gb[(long)tok * 2 * H + H + h];
    }
    double run = there ? (double)d_low : 1.;       // (a token that is not there decays nothing and writes nothing)
    const double beta_low = there ? (double)b_low : 0.;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      runs[wave][p][low] = run;
      const double before = __shfl(run, lane - (1 << p), kWave);
      run *= low >= 1 << p ? before : 1.;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    auto decays = [&](int upto, int count) {       // of the `count` tokens up to `upto`
      double d = 1.;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const bool on = count >> p & 1;
        const double v = runs[wave][p][max(upto, 0)];
        d *= on ? v : 1.;
        upto -= on ? 1 << p : 0;
      }
      return d;
    };
    float* f = of_sixteen + (long)G * 3 * T * ROWS + (long)h * kHeadFactors;
    if (high == 0) *reinterpret_cast<float2*>(f + 2 * T * T + 2 * low) = float2{(float)run, (float)decays(T - 1, T - 1 - low)};
    kk = part[0][0][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) kk += part[0][w][lane];
    qk = part[1][0][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) qk += part[1][w][lane];
    doublex4 L, LT, R;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * e + high, late = max(i, low);
      const double between = decays(late, late - min(i, low)), beta = __shfl(beta_low, late, kWave);
      double v = beta * between * kk[e];
      if (!(fabs(v) < (double)INFINITY)) v = 0.;   // (x of a token that is not finite is not either: it needs no help from M)
      L[e] = low < i ? v : 0.;
      LT[e] = low > i ? v : 0.;
      R[e] = (low == i ? 1. : 0.) - L[e];
      f[T * T + low % 4 * 4 * T + low / 4 * T + i] = low <= i ? (float)(between * qk[e]) : 0.f;
    }
    const doublex4 zero = {0., 0., 0., 0.};
    const doublex4 L2 = mul(LT, L, zero), L2T = mul(L, LT, zero);
    R = mul(L2T, R, R);
    const doublex4 L4 = mul(L2T, L2, zero), L4T = mul(L2, L2T, zero);
    R = mul(L4T, R, R);
    R = mul(mul(L4, L4T, zero), R, R);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[low / 4 * 4 * T + (4 * e + high) * 4 + low % 4] = (float)(R[e] * beta_low);
    __builtin_amdgcn_wave_barrier();
  }
}

// Workgroup (span, head, 16 columns), four waves: wave w holds the state's rows 64 c + 16 w ... + 15 as the results of
// the 32-bit matrix instruction 16 x 16 x 4 (rows 4 (lane / 16) + e, column lane % 16), which are its right operands too:
// which row a product covers is free.  The sums over the rows meet in LDS once a sixteen; x, u and the factors' products are
// every wave's own, the outputs' are shared out.  Operands come from memory two sixteens ahead, in whole kilobytes; values
// of tokens that are not there are out of a buffer's range: zeros.
template <int NB>
__global__ __launch_bounds__(kRecThreads, NB <= 3 ? 2 : 1) void gated_delta_sixteens_kernel(
    const float* __restrict__ vv, const float* __restrict__ factors, float* __restrict__ o_out,
    float* __restrict__ state, long slot_stride, const int* __restrict__ slots, const int* __restrict__ span_start,
    const int* __restrict__ span_pos, int H, int G, int dk, int dv, const ConvTail tail) {
  constexpr int WAVES = kRecThreads / kWave, T = kSixteen, ROWS = 64 * NB;
  __shared__ floatx4 met[2][WAVES][kWave];           // the waves' shares of S^T k
  __shared__ float outs[2][WAVES][4][kWave];         // and of the outputs
  __shared__ float slow[WAVES][T][T + 1];
  const int span = blockIdx.x, h = blockIdx.y, lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = h / (H / G), low = lane % 16, high = lane / 16;
  const int j = blockIdx.z * 16 + low;
  const long t0 = span_start[span];
  const int len = (int)(span_start[span + 1] - t0);
  const bool fresh = span_pos[span] == 0;
  float* S = state + (long)slots[span] * slot_stride + (long)h * dk * dv;
  floatx4 s[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 64 * c + 16 * wave + 4 * high + e;
      s[c][e] = (j < dv && r < dk && !fresh) ? S[(long)r * dv + j] : 0.f;
    }
  conv_tail_of_span(tail, slot_stride, slots[span], t0, t0 + len, fresh);
  const int HV = H * dv;
  auto range = [&](const float* base) {              // the span's rows, dv numbers of the last one
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, len > 0 ? (int)((((long)len - 1) * HV + dv) * 4) : 0, 0x00020000);
  };
  const auto v_rows = range(vv + t0 * HV + (long)h * dv), o_rows = range(o_out + t0 * HV + (long)h * dv);
  constexpr unsigned kNowhere = 0x80000000u;         // out of every range (see the host's check)
  const unsigned v_at = j < dv ? (unsigned)(4 * high * HV + j) * 4 : kNowhere;
  const unsigned o_at = j < dv ? (unsigned)((4 * high + wave) * HV + j) * 4 : kNowhere;
  const long stride = sixteen_floats(H, G, ROWS);
  const float* of_span = factors + (t0 / T + span) * stride;
  const float* of_keys = of_span + (long)g * 3 * T * ROWS;
  const float* of_head = of_span + (long)G * 3 * T * ROWS + (long)h * kHeadFactors;
  const int last = len > 0 ? (len - 1) / T : 0;
  auto f32 = [](unsigned x) { return __builtin_bit_cast(float, x); };
  struct Operands {
    floatx4 k[NB], q[NB], kt[NB], v, m;
    float b, all, upto, behind;                      // (decays: of token 4 high + lane % 4)
  };
  // The operands of the sixteen at t, a piece at a time, to be asked for between the products.  (Of a sixteen behind the
  // last one: the last one's again, not used.)
  constexpr int PIECES = 3 * NB + 8;
  auto ask = [&](int piece, int t, Operands& P) {
    const long at = min(t / T, last) * stride;
    auto four = [](const float* p) { return *reinterpret_cast<const floatx4*>(p); };
    const int quad = 4 * wave + high;
    if (piece < NB) {
      P.k[piece] = four(of_keys + at + ((quad + 16 * piece) * T + low) * 4);
    } else if (piece < 2 * NB) {
      P.q[piece - NB] = four(of_keys + at + T * ROWS + ((quad + 16 * (piece - NB)) * T + low) * 4);
    } else if (piece == 2 * NB) {
      const float2 d = *reinterpret_cast<const float2*>(of_head + at + 2 * T * T + 2 * (4 * high + lane % 4));
      P.upto = d.x;
      P.behind = d.y;
    } else if (piece < 2 * NB + 5) {
      const unsigned e = piece - 2 * NB - 1;
      P.v[e] = f32(__builtin_amdgcn_raw_buffer_load_b32(v_rows, v_at + ((unsigned)t + e) * HV * 4, 0, 0));
    } else if (piece == 2 * NB + 5) {
      P.m = four(of_head + at + (high * T + low) * 4);
    } else if (piece == 2 * NB + 6) {
      P.b = of_head[at + T * T + (wave * 4 + high) * T + low];
    } else if (piece < 3 * NB + 7) {
      const int c = piece - 2 * NB - 7;
      P.kt[c] = four(of_keys + at + 2 * T * ROWS + (high * ROWS + 64 * c + 16 * wave + low) * 4);
    } else {
      P.all = of_head[at + 2 * T * T + 2 * (T - 1)];
    }
  };
  auto mfma = [](float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
  auto lds_barrier = [&]() {   // orders LDS traffic only: loads from memory stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto write_out = [&](int t, int buf) {             // tokens t + 4 high + wave
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += outs[buf][w][wave][lane];
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o), o_rows, o_at + (unsigned)t * HV * 4, 0, 0);
  };
  // The sixteen at t; meanwhile the operands of the one at `then` are asked for.
  auto sixteen = [&](const Operands& P, int t, int buf, Operands& next, int then) {
    constexpr int FIRST = (NB + 1) / 2;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    int piece = 0;
    auto feed = [&]() {
      if (piece < PIECES) ask(piece++, then, next);
      __builtin_amdgcn_sched_barrier(0);
    };
    floatx4 a[NB], o[NB];                            // (a chain of sixteen products each: the sums' error, not their time)
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      a[c] = zero;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[c] = mfma(P.k[c][e], s[c][e], a[c]);
        feed();
      }
    }
#pragma unroll
    for (int c = 1; c < NB; ++c) a[0] += a[c];
    met[buf][wave][lane] = a[0];
    __builtin_amdgcn_sched_barrier(0);
    auto queries = [&](int c) {
      o[c] = zero;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[c] = mfma(P.q[c][e], s[c][e], o[c]);
        feed();
      }
    };
#pragma unroll
    for (int c = 0; c < FIRST; ++c) queries(c);      // while the sums are on their way
    lds_barrier();
    floatx4 x = met[buf][0][lane], others[WAVES - 1];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) others[w - 1] = met[buf][w][lane];
    if (t > 0) write_out(t - T, buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = FIRST; c < NB; ++c) queries(c);
    floatx4 upto, behind;
    upto[0] = dpp_moved<0x00>(P.upto), upto[1] = dpp_moved<0x55>(P.upto);      // (a four's lane 0, 1, 2, 3 to all of it)
    upto[2] = dpp_moved<0xAA>(P.upto), upto[3] = dpp_moved<0xFF>(P.upto);
    behind[0] = dpp_moved<0x00>(P.behind), behind[1] = dpp_moved<0x55>(P.behind);
    behind[2] = dpp_moved<0xAA>(P.behind), behind[3] = dpp_moved<0xFF>(P.behind);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) x += others[w - 1];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = fmaf(-upto[e], x[e], P.v[e]);
    floatx4 u = zero;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u = mfma(P.m[e], x[e], u);
      feed();
    }
#pragma unroll
    for (int c = 1; c < NB; ++c) o[0] += o[c];
    floatx4 out = o[0] * upto;
    const bool odd = !(fabsf(u[0]) < INFINITY && fabsf(u[1]) < INFINITY && fabsf(u[2]) < INFINITY && fabsf(u[3]) < INFINITY);
    if (__builtin_expect(__any(odd), 0)) {
      // A token that is not finite is to leave those before it alone: products with the zeros above the diagonals are
      // left out, and tokens that are not there write nothing.
      const float* f = of_head + t / T * stride;
#pragma unroll
      for (int e = 0; e < 4; ++e) slow[wave][4 * high + e][low] = x[e];
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * high + e;
        float v = 0.f;
        for (int l = 0; l <= i; ++l) v = fmaf(f[(l / 4 * T + i) * 4 + l % 4], slow[wave][l][low], v);
        if (t + i >= len) v = 0.f;
        if (e == 0) u[0] = v; else if (e == 1) u[1] = v; else if (e == 2) u[2] = v; else u[3] = v;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int e = 0; e < 4; ++e) slow[wave][4 * high + e][low] = u[e];
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * high + e;
        float v = 0.f;
        for (int l = wave; l <= i; l += 4) v = fmaf(f[T * T + (l % 4 * 4 + l / 4) * T + i], slow[wave][l][low], v);
        if (e == 0) out[0] += v; else if (e == 1) out[1] += v; else if (e == 2) out[2] += v; else out[3] += v;
      }
      __builtin_amdgcn_wave_barrier();
    } else {
      out = mfma(P.b, wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3], out);
    }
    u *= behind;
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      floatx4 more = zero;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        more = mfma(P.kt[c][e], u[e], more);
        feed();
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) s[c][e] = fmaf(P.all, s[c][e], more[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) outs[buf][wave][e][lane] = out[e];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) feed();
  };
  Operands P[3];                                     // (two sixteens ahead)
#pragma unroll
  for (int i = 0; i < PIECES; ++i) ask(i, 0, P[0]);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) ask(i, T, P[1]);
  int t = 0, buf = 0;
  for (; t + 2 * T < len; t += 3 * T, buf ^= 1) {    // (three a turn: operands in three sets of registers)
    sixteen(P[0], t, buf, P[2], t + 2 * T);
    sixteen(P[1], t + T, buf ^ 1, P[0], t + 3 * T);
    sixteen(P[2], t + 2 * T, buf, P[1], t + 4 * T);
  }
  if (t < len) sixteen(P[0], t, buf, P[2], t + 2 * T);
  if (t + T < len) sixteen(P[1], t + T, buf ^ 1, P[0], t + 3 * T);
  lds_barrier();
  if (len > 0) write_out((len - 1) / T * T, (len - 1) / T & 1);
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 64 * c + 16 * wave + 4 * high + e;
      if (j < dv && r < dk) S[(long)r * dv + j] = s[c][e];
    }
}

// ---------------------------------------------------------------------------- gated linear recurrence

constexpr int kGateTile = 16;                 // tokens, and output channels, of a matrix instruction
constexpr int kGateChunk = 1024;              // inputs of a block that LDS holds at a time

// proj: [nsplit][n][2 W], columns y | x.  Workgroup (NT tiles of 16 tokens, block b of the gates, OW times
// 16 of its output channels): the convolved inputs of the block's channels for its tokens go into LDS
// [tokens][inputs + 4], 1,024 inputs at a time; the gates' products run on the 32-bit matrix instruction 16x16x4 (an
// FMA chain).  The gates' matrices are read [block][in][out]: a lane's output channel is its
// lane % 16, so that a load reads 64 bytes of each of four rows.  A = inputs: lane l holds token l % 16,
// inputs 16 s + 4 (l / 16) + e of step s, e the instruction; which input a product covers is free as
// long as both operands agree, so a lane reads four with one 16-byte LDS read.  A sum's products go in chains of 64
// inputs that are added one after the other, as with the four threads to an output before: one chain of a block's 256
// left 1.3 times their error against 64 bits in the added terms (1.54e-7 against 1.18e-7 relative).
// KS waves share an output's inputs and meet in LDS: where there is one tile of tokens (a decode batch)
// the matrices' way from memory bounds the time, and it needs workgroups (16 channels each) and short
// chains; a prompt has tiles enough and is bound by its products.
// 1,500 tokens x 2,048 channels in blocks of 256: 140 -> 63 us (FMA on eight tokens at a time, 790 MB of matrices
// through L2) -> 56; 8 tokens: 18 -> 11 us, in a step, where the matrices come from memory, 28.8 -> 16.9 (32 workgroups then, 128 now) -> 14.0 -> 10.0: a
// run's inputs are now asked for together whatever the number of the projection's slices (a loop over them for every input waited eleven
// times), the tokens' spans, the gates' constants and the matrices in one go before anything is waited for, and the arguments they need
// come with the launch.
// TAPS: the convolution's where it is 4, 8 for any number up to 8, 0 for more.  ONE: a block's inputs fit into LDS at
// once; the sums then begin behind the convolution and take no registers in it (72 instead of 89, three workgroups a CU).
template <int NT, int KS, int OW, int TAPS, bool ONE>
__global__ __launch_bounds__(kWave * KS * OW) void linear_recurrence_prep_kernel(
    const int* __restrict__ span_of_token, const int* __restrict__ span_start, const int* __restrict__ slots, const int* __restrict__ span_pos,
    const float* __restrict__ proj, int n, int W, int bs, int taps, const float* __restrict__ conv_w, const float* __restrict__ conv_b,
    int nsplit, const float* __restrict__ x_bias, const float* __restrict__ wr_t, const float* __restrict__ wi_t, long split_stride,
    const float* __restrict__ state, long slot_stride, const float* __restrict__ br, const float* __restrict__ bi, const float* __restrict__ rate,
    float* __restrict__ a_out, float* __restrict__ b_out) {
  constexpr int TT = NT * kGateTile, THREADS = kWave * KS * OW;
  extern __shared__ __attribute__((aligned(16))) float us[];
  const int b = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int chunk = min((bs + 15) / 16 * 16, kGateChunk), ld = chunk + 4;      // inputs in LDS at a time
  const long tfirst = (long)blockIdx.x * TT;
  const int nt = (int)min((long)TT, n - tfirst);
  const long cols = 2L * W;
  const int ks = wave % KS, ow = wave / KS;
  const int col = lane % 16, quad = lane / 16;
  const int o = (blockIdx.z * OW + ow) * kGateTile + col;
  const int oc = min(o, bs - 1);
  const float* wr = wr_t + (long)b * bs * bs;
  const float* wi = wi_t + (long)b * bs * bs;
  struct Pair { float r[4], i[4]; };
  auto fetch = [&](int first) -> Pair {       // (inputs that do not exist: zeros, whatever the last row holds)
    Pair P;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int in = first + 4 * quad + e;
      const unsigned at = (unsigned)min(in, bs - 1) * bs + oc;      // (blocks of up to 4,096 channels)
      const float r = wr[at], g = wi[at];
      P.r[e] = in < bs ? r : 0.f;
      P.i[e] = in < bs ? g : 0.f;
    }
    return P;
  };
  floatx4 ar[NT], ai[NT], own[NT];            // own: the outputs' own inputs
#pragma unroll
  for (int t = 0; t < NT; ++t) ar[t] = ai[t] = own[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  constexpr int CHAIN = 4;                    // steps of a chain
  constexpr int AHEAD = KS > 1 ? CHAIN : 1;   // steps asked for ahead
  __shared__ int4 spans[TT];                  // the tokens' spans
  // A decode batch asks for the tokens' spans first and, before it waits for them, for all that needs none of them.
  constexpr bool AT_ONCE = KS > 1 && TAPS > 1;
  const int span = span_of_token[tfirst + min(tid, nt - 1)];
  float rb = 0.f, ib = 0.f, rt = 0.f;
  auto constants = [&] {
    const int c = b * bs + oc;
    rb = br[c], ib = bi[c], rt = rate[c];
  };
  if (AT_ONCE) {
    asm volatile("" ::"s"(conv_w), "s"(conv_b), "s"(nsplit), "s"(x_bias), "s"(wr_t), "s"(wi_t), "s"(state), "s"(slot_stride), "s"(br), "s"(bi),
                 "s"(rate), "s"(a_out), "s"(b_out));
    constants();
  }
  const int4 mine = int4{span_start[span], slots[span], span_pos[span] == 0, 0};
  int k0 = 0;
  do {
    if (!ONE && k0 > 0) __syncthreads();
    const int steps = (min(chunk, bs - k0) + 15) / 16;
    const int per = (steps + KS - 1) / KS, s0 = ks * per, s1 = min(steps, s0 + per);
    // The first of this wave's share of the matrices: a decode batch's whole chain (they come from memory, and nothing
    // in them waits for the convolution), a prompt's first step.
    Pair w[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (KS > 1) w[i] = fetch(k0 + 16 * min(s0 + i, steps - 1));
    if (k0 == 0) {
      if (tid < nt) spans[tid] = mine;
      __syncthreads();
    }
    if (TAPS > 0 && (nt > 1 || KS > 1)) {
      // A thread takes a channel for a run of RUN tokens and asks for the run's inputs at once, each
      // for all the taps it meets, instead of for every tap of every token on its own.
      constexpr int MOST = TAPS > 0 ? TAPS : 1, RUN = 8;
      const int K = TAPS == 4 ? 3 : taps - 1;
      for (int i = tid; i < TT / RUN * chunk; i += THREADS) {
        const int r = i / chunk, e = k0 + i - r * chunk, c = b * bs + e, tt0 = r * RUN;
        const bool there = e < bs && tt0 < nt;
        float x[RUN + MOST - 1], wt[MOST];
        const int cc = min(c, W - 1);
        if (there) {
          auto row_at = [&](int q) { return proj + (long)min(max((int)tfirst + tt0 - K + q, 0), n - 1) * cols + W + cc; };
#pragma unroll
          for (int q = 0; q < RUN + MOST - 1; ++q) {        // (rows that are not there: some row that is, not used)
            if (q >= RUN + K) break;
            x[q] = *row_at(q);
          }
#pragma unroll
          for (int j = 0; j < MOST; ++j) wt[j] = conv_w[(long)c * taps + min(j, K)];
          for (int sp = 1; sp < nsplit; ++sp)
#pragma unroll
            for (int q = 0; q < RUN + MOST - 1; ++q) {
              if (q >= RUN + K) break;
              x[q] += row_at(q)[sp * split_stride];
            }
        }
        const float cb = there ? conv_b[c] : 0.f, xb = there && x_bias ? x_bias[c] : 0.f;
        int4 sp[RUN];                                       // first row, slot, whether the span starts at position 0
#pragma unroll
        for (int q = 0; q < RUN; ++q) sp[q] = spans[min(tt0 + q, nt - 1)];
        // A decode batch's tokens are spans of their own and find all but one input in the requests' states: a run of
        // tokens with a span's start in it asks for all their entries at once (in a prompt, where such runs are few, one by one: the
        // entries' registers would cost a workgroup a CU).
        float st[AT_ONCE ? RUN : 1][AT_ONCE ? TAPS - 1 : 1];
        if constexpr (AT_ONCE) {
          bool starts = false;
#pragma unroll
          for (int q = 0; q < RUN; ++q) starts |= (int)tfirst + min(tt0 + q, nt - 1) - K < sp[q].x;
          if (starts && there) {
#pragma unroll
            for (int q = 0; q < RUN; ++q) {                 // (tokens that are not there: the last one's, not used)
              const float* from = state + (long)sp[q].y * slot_stride + (long)c * K;
#pragma unroll
              for (int j = 0; j < TAPS - 1; ++j) st[q][j] = from[min(j, K - 1)];
            }
          }
        }
        if (x_bias)                                         // the convolution's input carries the projection's bias
#pragma unroll
          for (int q = 0; q < RUN + MOST - 1; ++q) x[q] += xb;
#pragma unroll
        for (int q = 0; q < RUN; ++q) {
          float v = 0.f;
          if (there && tt0 + q < nt) {
            const int t = (int)tfirst + tt0 + q;
#pragma unroll
            for (int j = 0; j < MOST; ++j) {
              if (j > K) break;
              const int back = t - K + j - sp[q].x;         // rows behind the span's first
              float in = x[q + j];
              if constexpr (AT_ONCE) {
                float was = st[q][0];                       // entry K + back, by choice: the entries stay in registers
#pragma unroll
                for (int i = 1; i < TAPS - 1; ++i) was = i == K + back ? st[q][i] : was;
                in = back < 0 ? (sp[q].z ? 0.f : was) : in;
              } else if (back < 0) {
                in = sp[q].z ? 0.f : state[(long)sp[q].y * slot_stride + (long)c * K + K + back];
              }
              v = fmaf(wt[j], in, v);
            }
            v += cb;
          }
          us[(tt0 + q) * ld + e - k0] = v;
        }
      }
    } else {
      for (int i = tid; i < TT * chunk; i += THREADS) {
        const int tt = i / chunk, e = k0 + i - tt * chunk, c = b * bs + e;
        float v = 0.f;
        if (tt < nt && e < bs) {
          const int4 sp = spans[tt];
          // (the convolution's input carries the projection's bias; before position 0 it is zero)
          v = conv_at(proj, nsplit, split_stride, cols, W + c, x_bias - W, conv_w + (long)c * taps, taps,
                      state + (long)sp.y * slot_stride + (long)c * (taps - 1), sp.z != 0, tfirst + tt, sp.x) + conv_b[c];
        }
        us[tt * ld + e - k0] = v;
      }
    }
    if (KS == 1) w[0] = fetch(k0 + 16 * min(s0, steps - 1));
    __syncthreads();
    if (o >= k0 && o < k0 + chunk)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) own[t][i] = us[(t * kGateTile + 4 * quad + i) * ld + o - k0];
    for (int c0 = s0; c0 < s1; c0 += CHAIN) {
      floatx4 cr[NT], ci[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) cr[t] = ci[t] = floatx4{0.f, 0.f, 0.f, 0.f};
      auto step = [&](int s, const Pair& w) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const floatx4 u = *reinterpret_cast<const floatx4*>(&us[(t * kGateTile + col) * ld + 16 * s + 4 * quad]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            cr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[e], w.r[e], cr[t], 0, 0, 0);
            ci[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[e], w.i[e], ci[t], 0, 0, 0);
          }
        }
      };
      if constexpr (KS > 1) {
#pragma unroll
        for (int i = 0; i < CHAIN; ++i)
          if (c0 + i < s1) step(c0 + i, w[i]);
        if (c0 + CHAIN < s1)
#pragma unroll
          for (int i = 0; i < CHAIN; ++i) w[i] = fetch(k0 + 16 * min(c0 + CHAIN + i, steps - 1));
      } else {
#pragma unroll 1
        for (int s = c0; s < min(s1, c0 + CHAIN); ++s) {
          const Pair next = fetch(k0 + 16 * min(s + 1, steps - 1));
          step(s, w[0]);
          w[0] = next;
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        ar[t] += cr[t];
        ai[t] += ci[t];
      }
    }
    k0 += chunk;
  } while (!ONE && k0 < bs);
  if constexpr (KS > 1) {                     // the waves' shares, in a fixed order
    static_assert(OW == 1 && NT == 1, "one tile a workgroup");
    __shared__ floatx4 red[KS - 1][2][kWave];
    if (ks > 0) {
      red[ks - 1][0][lane] = ar[0];
      red[ks - 1][1][lane] = ai[0];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int q = 0; q < KS - 1; ++q) {
      ar[0] += red[q][0][lane];
      ai[0] += red[q][1][lane];
    }
  }
  if (o >= bs) return;
  const int c = b * bs + o;
  if (!AT_ONCE) constants();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {             // D[token 4 quad + i][output lane % 16]
      const int tt = t * kGateTile + 4 * quad + i;
      if (tt >= nt) continue;
      const float r = sigmoid_f32(ar[t][i] + rb), ig = sigmoid_f32(ai[t][i] + ib);
      const float log_a = -rt * r;
      const float a = expf(log_a);
      const float mult = sqrtf(fmaxf(-expm1f(2.f * log_a), 0.f));      // sqrt(1 - a^2)
      a_out[(tfirst + tt) * W + c] = a;
      b_out[(tfirst + tt) * W + c] = mult * ig * own[t][i];
    }
}

template <int NT, int KS, int OW, int TAPS, bool ONE>
static int recurrence_prep_launch_chunks(const float* proj, int nsplit, long split_stride, const float* x_bias,
                                  const float* conv_w, const float* conv_b, int taps, const float* state,
                                  long slot_stride, const float* wr_t, const float* wi_t, const float* br,
                                  const float* bi, const float* rate, const int* span_of_token, const int* slots,
                                  const int* span_start, const int* span_pos, float* a_out, float* b_out, int n, int W,
                                  int blocks, hipStream_t stream) {
  const int bs = W / blocks;
  const int chunk = ceil_div(bs, 16) * 16 < kGateChunk ? ceil_div(bs, 16) * 16 : kGateChunk;
  const size_t lds = (size_t)NT * kGateTile * (chunk + 4) * sizeof(float);
  static size_t raised_to = 48 * 1024;      // beside the kernel's own LDS
  if (lds > raised_to) {
    (void)hipFuncSetAttribute((const void*)linear_recurrence_prep_kernel<NT, KS, OW, TAPS, ONE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    raised_to = lds;
  }
  hipLaunchKernelGGL((linear_recurrence_prep_kernel<NT, KS, OW, TAPS, ONE>),
                     dim3(ceil_div(n, NT * kGateTile), blocks, ceil_div(bs, OW * kGateTile)), dim3(kWave * KS * OW), lds,
                     stream, span_of_token, span_start, slots, span_pos, proj, n, W, bs, taps, conv_w, conv_b, nsplit, x_bias, wr_t, wi_t,
                     split_stride, state, slot_stride, br, bi, rate, a_out, b_out);
  KLLM_CHECK_LAUNCH("linear_recurrence_prep");
  return 0;
}

template <int NT, int KS, int OW, int TAPS, typename... A>
static int recurrence_prep_launch(int bs, A... args) {
  return bs <= kGateChunk ? recurrence_prep_launch_chunks<NT, KS, OW, TAPS, true>(args...)
                          : recurrence_prep_launch_chunks<NT, KS, OW, TAPS, false>(args...);
}

// S <- a S + b along a span; out = S * gelu_tanh(y + y_bias).  Eight tokens' numbers are asked
// for at a time, so that the chain holds arithmetic only.
// A span's tokens are cut into SEGS segments: S_t = a_t S_(t-1) + b_t is a composition of maps
// S -> a S + b, and so is a whole segment's (A S + B, with A the product of its a and B its own chain
// from zero).  Every segment's threads first run its chain from zero, the segments' (A, B) meet in LDS,
// those before a segment are folded into its starting state and it runs once more, now writing.  A
// chain of n steps becomes two of n / SEGS.
// CH channels and SEGS segments a workgroup (see kllm_linear_recurrence_scan); a span of up to LEAST tokens is one
// segment, and the others' threads leave at once.  The convolution's inputs are left by workgroups of their own, behind those of
// a span's channels: in front of a chain they held it up (us, before and now, 2,048 channels: 480 tokens beside 20 single ones 23.1 / 17.1,
// 1,500 tokens 36.0 / 31.9, 8 single tokens 5.2 / 4.5).  Where single tokens have twelve workgroups a CU the chain's threads do it, as
// before (64 tokens, 4,096 channels: 8.2 us; 8.9 with workgroups of their own; at 2,048 channels 6.5 and 6.3).
template <typename T, int CH, int SEGS>
__global__ __launch_bounds__(CH * SEGS) void linear_recurrence_scan_kernel(
    const int* __restrict__ span_start, const int* __restrict__ slots, const int* __restrict__ span_pos, const float* __restrict__ a_in,
    const float* __restrict__ b_in, const float* __restrict__ proj, int W, int nsplit, long split_stride, const float* __restrict__ y_bias,
    float* __restrict__ state, long slot_stride, T* __restrict__ out, const ConvTail tail) {
  __shared__ float seg_a[SEGS][CH], seg_b[SEGS][CH];
  int at = blockIdx.y;                                    // (vector loads: scalar ones come one behind the other)
  asm volatile("" : "+v"(at));
  const int first_v = span_start[at], last_v = span_start[at + 1], slot_v = slots[at], pos_v = span_pos[at];
  asm volatile("" ::"s"(split_stride), "s"(y_bias), "s"(state), "s"(slot_stride), "s"(out));
  const int lane = threadIdx.x % CH, seg = threadIdx.x / CH;
  const int c = min((int)blockIdx.x * CH + lane, W - 1);
  const bool ok = blockIdx.x * CH + lane < W;
  const float yb = y_bias[c];
  const int t0 = __builtin_amdgcn_readfirstlane(first_v), t1 = __builtin_amdgcn_readfirstlane(last_v), slot = __builtin_amdgcn_readfirstlane(slot_v);
  const bool fresh = __builtin_amdgcn_readfirstlane(pos_v) == 0;
  const int own = (W + CH - 1) / CH;                      // workgroups of the chain
  if (SEGS == 1 && (int)gridDim.x == own && tail.taps > 1 && ok)
    conv_tail(tail, slot_stride, c, slot, t0, t1, fresh);
  if ((int)blockIdx.x >= own) {
    const int cc = ((int)blockIdx.x - own) * CH * SEGS + (int)threadIdx.x;
    if (cc < W) conv_tail(tail, slot_stride, cc, slot, t0, t1, fresh);
    return;
  }
  const int len = t1 - t0;
  constexpr int U = 8, LEAST = 4;                         // tokens asked for at a time, of a segment at least
  const int per = SEGS > 1 ? max(LEAST, (len + SEGS - 1) / SEGS) : len;
  const bool cut = SEGS > 1 && len > LEAST;
  const int a0 = min(t1, t0 + seg * per), a1 = min(t1, a0 + per);
  float* st = state + (long)slot * slot_stride + c;
  if (!cut && seg > 0) return;                            // (nobody meets)
  float S = fresh ? 0.f : *st;
  if (cut) {
    float A = 1.f, B = 0.f;
    for (int tb = a0; tb < a1; tb += U) {
      float a[U], b[U];
#pragma unroll
      for (int q = 0; q < U; ++q) {
        const long t = min(tb + q, a1 - 1);
        a[q] = a_in[t * W + c];
        b[q] = b_in[t * W + c];
      }
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (tb + q >= a1) break;
        B = fmaf(a[q], B, b[q]);
        A *= a[q];
      }
    }
    seg_a[seg][lane] = A;
    seg_b[seg][lane] = B;
    __syncthreads();
#pragma unroll 8
    for (int s = 0; s < seg; ++s) S = fmaf(seg_a[s][lane], S, seg_b[s][lane]);
  }
  // A slice of eight tokens' branches together (in a loop over the slices for every token each waited for its load: 1,500 tokens of 2,048 channels
  // 33.4 -> 31.6 us, a prompt of 200 at Natenex sizes 1,239 -> 1,220, a step of 8 tokens 556 -> 552), the activation only of
  // tokens that are there; a span of its own channels asks for no token that is not.
  for (int tb = a0; tb < a1; tb += U) {
    float a[U], b[U], y[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      if (SEGS == 1 && q > 0 && tb + q >= a1) break;
      const long t = min(tb + q, a1 - 1);
      a[q] = a_in[t * W + c];
      b[q] = b_in[t * W + c];
      y[q] = proj[t * 2 * W + c];
    }
    for (int s = 1; s < nsplit; ++s)
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (SEGS == 1 && q > 0 && tb + q >= a1) break;
        y[q] += proj[s * split_stride + (long)min(tb + q, a1 - 1) * 2 * W + c];
      }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      if (tb + q >= a1) break;
      S = fmaf(a[q], S, b[q]);
      const float gate = gate_act<T>(y[q] + yb, ACT_GELU_TANH);
      if (ok) out[(long)(tb + q) * W + c] = from_f32<T>(S * gate);
    }
  }
  // the last segment ends at the span's last token (an empty one has folded all); every segment has
  // read the state by then: they met behind it
  if (ok && seg == (cut ? SEGS - 1 : 0)) *st = S;
}

// out = sa * (sum of a's slices) + sb * (sum of b's slices), element by element.
__global__ void scaled_sum_kernel(float* __restrict__ out, const float* __restrict__ a, int na, long stride_a, float sa,
                                  const float* __restrict__ b, int nb, long stride_b, float sb, long count) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float va = 0.f, vb = 0.f;
  for (int s = 0; s < na; ++s) va += a[i + s * stride_a];
  for (int s = 0; s < nb; ++s) vb += b[i + s * stride_b];
  out[i] = fmaf(sa, va, sb * vb);
}

// out = sa * wa * N(sum of a's slices) + sb * wb * N(sum of b's slices), row by row; N(v) = v /
// sqrt(mean(v^2) + eps).  One workgroup a row; both rows wait in LDS between the two passes.
__global__ __launch_bounds__(kRecThreads) void normed_sum_kernel(
    float* __restrict__ out, const float* __restrict__ a, int na, long stride_a, float sa, const float* __restrict__ wa,
    const float* __restrict__ b, int nb, long stride_b, float sb, const float* __restrict__ wb, int d, float eps) {
  extern __shared__ float rows_lds[];     // [2][d]
  __shared__ float red[16];
  const long r = blockIdx.x;
  float ssa = 0.f, ssb = 0.f;
  for (int i = threadIdx.x; i < d; i += kRecThreads) {
    float va = 0.f, vb = 0.f;
    for (int s = 0; s < na; ++s) va += a[r * d + i + s * stride_a];
    for (int s = 0; s < nb; ++s) vb += b[r * d + i + s * stride_b];
    rows_lds[i] = va;
    rows_lds[d + i] = vb;
    ssa = fmaf(va, va, ssa);
    ssb = fmaf(vb, vb, ssb);
  }
  const float ra = sa / sqrtf(block_sum(ssa, red) / (float)d + eps);
  const float rb = sb / sqrtf(block_sum(ssb, red) / (float)d + eps);
  for (int i = threadIdx.x; i < d; i += kRecThreads)     // a thread reads back what it wrote itself
    out[r * d + i] = fmaf(rows_lds[i] * ra, wa[i], rows_lds[d + i] * rb * wb[i]);
}

}  // namespace kllm

using namespace kllm;

extern "C" int kllm_normed_sum(float* out, const float* a, int na, long stride_a, float sa, const float* wa,
                               const float* b, int nb, long stride_b, float sb, const float* wb, int n, int d,
                               float eps, hipStream_t stream) {
  KLLM_REQUIRE(out && a && b && wa && wb && na >= 1 && nb >= 1 && n > 0 && d > 0, "normed_sum: null pointer or bad sizes");
  const size_t lds = 2 * (size_t)d * sizeof(float);
  KLLM_REQUIRE(lds <= 128 * 1024, "normed_sum: rows of %d do not fit into LDS", d);
  static size_t raised_to = 48 * 1024;
  if (lds > raised_to) {
    (void)hipFuncSetAttribute((const void*)normed_sum_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    raised_to = lds;
  }
  hipLaunchKernelGGL(normed_sum_kernel, dim3(n), dim3(kRecThreads), lds, stream, out, a, na, stride_a, sa, wa, b, nb,
                     stride_b, sb, wb, d, eps);
  KLLM_CHECK_LAUNCH("normed_sum");
  return 0;
}

extern "C" int kllm_scaled_sum(float* out, const float* a, int na, long stride_a, float sa, const float* b, int nb,
                               long stride_b, float sb, long count, hipStream_t stream) {
  KLLM_REQUIRE(out && a && b && na >= 1 && nb >= 1 && count > 0, "scaled_sum: null pointer or bad sizes");
  hipLaunchKernelGGL(scaled_sum_kernel, dim3(ceil_div(count, 256)), dim3(256), 0, stream, out, a, na, stride_a, sa, b, nb,
                     stride_b, sb, count);
  KLLM_CHECK_LAUNCH("scaled_sum");
  return 0;
}

extern "C" int kllm_conv_state_update(const float* proj, int nsplit, long split_stride, int cols, int col0, int C,
                                      const float* in_bias, float* state, long slot_stride, int taps, const int* slots,
                                      const int* span_start, const int* span_pos, int n_spans, hipStream_t stream) {
  KLLM_REQUIRE(proj && state && slots && span_start && span_pos, "conv_state_update: null pointer");
  KLLM_REQUIRE(nsplit >= 1 && cols > 0 && col0 >= 0 && C > 0 && col0 + C <= cols && n_spans > 0 && n_spans <= 65535,
               "conv_state_update: bad sizes cols=%d col0=%d C=%d spans=%d", cols, col0, C, n_spans);
  KLLM_REQUIRE(taps >= 1 && taps <= kMaxTaps, "conv_state_update: %d taps (1 to %d)", taps, kMaxTaps);
  if (taps == 1) return 0;
  const ConvTail tail = {proj, split_stride, cols, in_bias, state, nsplit, col0, C, taps};
  hipLaunchKernelGGL(conv_state_update_kernel, dim3(ceil_div(C, kRecThreads), n_spans), dim3(kRecThreads), 0, stream, tail,
                     slot_stride, slots, span_start, span_pos);
  KLLM_CHECK_LAUNCH("conv_state_update");
  return 0;
}

extern "C" int kllm_gated_delta_prep(const float* proj, int nsplit, long split_stride, const float* conv_w, int taps,
                                     const float* state, long slot_stride, const float* a_log, const float* dt_bias,
                                     const int* span_of_token, const int* slots, const int* span_start,
                                     const int* span_pos, float* qn, float* kn, float* vv, float* gb, float* gate,
                                     int n, int H, int G, int dk, int dv, float unit_eps, int cols,
                                     const float* a_sums, int a_ns, long a_stride, int a_row, const float* gate_sums,
                                     int g_ns, long g_stride, int g_row, int gate_sigmoid, float* dec,
                                     hipStream_t stream) {
  KLLM_REQUIRE(proj && conv_w && state && a_log && dt_bias && span_of_token && slots && span_start && span_pos && qn &&
                   kn && vv && gb && gate, "gated_delta_prep: null pointer");
  KLLM_REQUIRE((a_sums == nullptr) == (dec == nullptr) && (!a_sums || a_ns >= 1) && (!gate_sums || g_ns >= 1),
               "gated_delta_prep: decays per key channel come with their sums and a place for them");
  KLLM_REQUIRE(cols >= 2 * G * dk + H * dv + (a_sums ? H : 2 * H) + (gate_sums ? 0 : H * dv),
               "gated_delta_prep: %d columns do not hold the projections", cols);
  KLLM_REQUIRE(n > 0 && H > 0 && G > 0 && H % G == 0 && dk > 0 && dv > 0 && nsplit >= 1,
               "gated_delta_prep: bad sizes n=%d H=%d G=%d dk=%d dv=%d", n, H, G, dk, dv);
  KLLM_REQUIRE(taps >= 1 && taps <= kMaxTaps, "gated_delta_prep: %d taps (1 to %d)", taps, kMaxTaps);
  KLLM_REQUIRE(dk <= 4 * kWave, "gated_delta_prep: key heads of %d (up to %d)", dk, 4 * kWave);
  KLLM_REQUIRE((!a_sums || a_row >= H * dk) && (!gate_sums || g_row >= H * dv),
               "gated_delta_prep: rows of %d and %d sums do not hold the decays and the gates", a_row, g_row);
  const int items = 2 * G + H, per_wg = kRecThreads / kWave;
  KLLM_REQUIRE(ceil_div(items, per_wg) <= 65535, "gated_delta_prep: %d heads are too many for the grid", items);
#define KLLM_GDP(TAPS, R)                                                                                                                \
  hipLaunchKernelGGL((gated_delta_prep_kernel<TAPS, R>), dim3(n, ceil_div(items, per_wg)), dim3(kRecThreads), 0, stream, span_of_token,         \
                     span_start, span_pos, slots, proj, H, G, dk, dv, conv_w, taps, nsplit, (long)cols, split_stride, state, slot_stride,   \
                     a_log, dt_bias, qn, kn, vv, gb, gate, unit_eps, a_sums, a_ns, a_stride, (long)a_row, gate_sums, g_ns, g_stride,       \
                     (long)g_row, gate_sigmoid, dec)
#define KLLM_GDT(TAPS)                                                              \
  do {                                                                              \
    if (dk <= kWave && dv <= kWave) KLLM_GDP(TAPS, 1); else KLLM_GDP(TAPS, 2);       \
  } while (0)
  if (taps == 1) KLLM_GDT(1);
  else if (taps == 2) KLLM_GDT(2);
  else if (taps == 3) KLLM_GDT(3);
  else if (taps == 4) KLLM_GDT(4);
  else KLLM_GDP(0, 2);
#undef KLLM_GDT
#undef KLLM_GDP
  KLLM_CHECK_LAUNCH("gated_delta_prep");
  return 0;
}

extern "C" int kllm_gated_delta_max_dim(void) { return 16 * kDeltaParts; }

extern "C" int kllm_gated_delta_factor_floats(int H, int G, int dk) {
  if (H <= 0 || G <= 0 || dk <= 0 || dk > 16 * kDeltaParts) return -1;
  const long floats = sixteen_floats(H, G, ceil_div(dk, 64) * 64);
  return floats < 0x7fffffffL ? (int)floats : -1;
}

extern "C" int kllm_gated_delta_factors(const float* qn, const float* kn, const float* gb, const int* span_start,
                                        float* factors, int n, int n_spans, int H, int G, int dk, hipStream_t stream) {
  KLLM_REQUIRE(qn && kn && gb && span_start && factors, "gated_delta_factors: null pointer");
  KLLM_REQUIRE(n > 0 && n_spans > 0 && H > 0 && G > 0 && G <= 65535 && H % G == 0 && dk > 0 && dk <= 16 * kDeltaParts,
               "gated_delta_factors: bad sizes n=%d spans=%d H=%d G=%d dk=%d (keys of up to %d)", n, n_spans, H, G, dk,
               16 * kDeltaParts);
  KLLM_REQUIRE(((uintptr_t)factors & 15) == 0, "gated_delta_factors: the factors' place is not aligned to 16 bytes");
  const int nb = ceil_div(dk, 64);
  const bool v4 = dk % 4 == 0 && (((uintptr_t)qn | (uintptr_t)kn) & 15) == 0;
#define KLLM_GDF(NB, V4)                                                                                              \
  hipLaunchKernelGGL((gated_delta_factors_kernel<NB, V4>), dim3(ceil_div(n, kSixteen) + n_spans, G),                     \
                     dim3(kRecThreads), 0, stream, qn, kn, gb, span_start, factors, n_spans, H, G, dk)
#define KLLM_GDFN(NB)               \
  do {                              \
    if (v4) KLLM_GDF(NB, true);     \
    else KLLM_GDF(NB, false);       \
  } while (0)
  if (nb <= 1) KLLM_GDFN(1);
  else if (nb <= 2) KLLM_GDFN(2);
  else if (nb <= 3) KLLM_GDFN(3);
  else KLLM_GDFN(4);
#undef KLLM_GDFN
#undef KLLM_GDF
  KLLM_CHECK_LAUNCH("gated_delta_factors");
  return 0;
}

extern "C" int kllm_gated_delta_scan(const float* qn, const float* kn, const float* vv, const float* gb, float* o_out,
                                     float* state, long slot_stride, const int* slots, const int* span_start,
                                     const int* span_pos, int n, int n_spans, int H, int G, int dk, int dv,
                                     const float* dec, const float* factors, const float* conv_proj, int conv_nsplit,
                                     long conv_stride, int conv_cols, int conv_channels, float* conv_state, int taps,
                                     hipStream_t stream) {
  KLLM_REQUIRE(qn && kn && vv && gb && o_out && state && slots && span_start && span_pos,
               "gated_delta_scan: null pointer");
  KLLM_REQUIRE(n > 0 && n_spans > 0 && H > 0 && H <= 65535 && G > 0 && H % G == 0 && dk > 0 && dk <= 16 * kDeltaParts && dv > 0,
               "gated_delta_scan: bad sizes spans=%d H=%d G=%d dk=%d dv=%d (keys of up to %d)", n_spans, H, G, dk, dv,
               16 * kDeltaParts);
  KLLM_REQUIRE(!conv_state || (conv_proj && conv_nsplit >= 1 && conv_channels > 0 && conv_channels <= conv_cols &&
                               taps >= 1 && taps <= kMaxTaps),
               "gated_delta_scan: the convolution's inputs do not fit (%d channels of %d columns, %d taps)", conv_channels,
               conv_cols, taps);
  ConvTail tail = {conv_proj, conv_stride, conv_cols, nullptr, conv_state, conv_nsplit, 0, conv_channels, taps};
  if (!conv_state) tail.taps = 0;
  const dim3 grid(n_spans, H, ceil_div(dv, kDeltaCols));
  KLLM_REQUIRE(grid.z <= 65535, "gated_delta_scan: values too wide for the grid");
  const int nb = ceil_div(dk, 64);
  if (factors) {
    KLLM_REQUIRE(!dec, "gated_delta_scan: factors of tokens with decays per key channel");
    KLLM_REQUIRE(((long)n + 4 * kSixteen) * H * dv < 1L << 29, "gated_delta_scan: %d rows of %d values are beyond 2 GiB, not"
                 " built with factors", n, H * dv);
    KLLM_REQUIRE(((uintptr_t)factors & 15) == 0, "gated_delta_scan: the factors are not aligned to 16 bytes");
#define KLLM_GDX(NB)                                                                                                   \
  hipLaunchKernelGGL((gated_delta_sixteens_kernel<NB>), grid, dim3(kRecThreads), 0, stream, vv, factors, o_out, state, \
                     slot_stride, slots, span_start, span_pos, H, G, dk, dv, tail)
    if (nb <= 1) KLLM_GDX(1);
    else if (nb <= 2) KLLM_GDX(2);
    else if (nb <= 3) KLLM_GDX(3);
    else KLLM_GDX(4);
#undef KLLM_GDX
    KLLM_CHECK_LAUNCH("gated_delta_scan");
    return 0;
  }
#define KLLM_GDS(NB)                                                                                                   \
  do {                                                                                                                 \
    if (dec)                                                                                                           \
      hipLaunchKernelGGL((gated_delta_scan_kernel<NB, true>), grid, dim3(kRecThreads), 0, stream, span_start, slots,         \
                         span_pos, state, H, G, dk, dv, slot_stride, kn, qn, vv, gb, o_out, dec, tail);                \
    else                                                                                                               \
      hipLaunchKernelGGL((gated_delta_scan_kernel<NB, false>), grid, dim3(kRecThreads), 0, stream, span_start, slots,        \
                         span_pos, state, H, G, dk, dv, slot_stride, kn, qn, vv, gb, o_out, dec, tail);                \
  } while (0)
  if (nb <= 1) KLLM_GDS(1);
  else if (nb <= 2) KLLM_GDS(2);
  else if (nb <= 3) KLLM_GDS(3);
  else KLLM_GDS(4);
#undef KLLM_GDS
  KLLM_CHECK_LAUNCH("gated_delta_scan");
  return 0;
}

extern "C" int kllm_linear_recurrence_prep(const float* proj, int nsplit, long split_stride, const float* x_bias,
                                           const float* conv_w, const float* conv_b, int taps, const float* state,
                                           long slot_stride, const float* wr_t, const float* wi_t, const float* br,
                                           const float* bi, const float* rate, const int* span_of_token,
                                           const int* slots, const int* span_start, const int* span_pos, float* a_out,
                                           float* b_out, int n, int W, int blocks, hipStream_t stream) {
  KLLM_REQUIRE(proj && x_bias && conv_w && conv_b && state && wr_t && wi_t && br && bi && rate && span_of_token &&
                   slots && span_start && span_pos && a_out && b_out, "linear_recurrence_prep: null pointer");
  KLLM_REQUIRE(n > 0 && W > 0 && blocks > 0 && blocks <= 65535 && W % blocks == 0 && nsplit >= 1,
               "linear_recurrence_prep: bad sizes n=%d W=%d blocks=%d", n, W, blocks);
  KLLM_REQUIRE(taps >= 1 && taps <= kMaxTaps, "linear_recurrence_prep: %d taps (1 to %d)", taps, kMaxTaps);
  const int bs = W / blocks;
  KLLM_REQUIRE(bs <= 4096, "linear_recurrence_prep: blocks of %d channels (up to 4,096)", bs);
  // A decode batch shares a sum's inputs out over four waves and takes 16 channels a workgroup: short chains, and
  // workgroups enough.  The workgroups of a block repeat its convolution and each tile of tokens reads the matrices
  // again, so that from three workgroups a CU on (or what LDS lets run side by side) eight waves take 16 channels each, and two tiles of
  // tokens at a time once those give every CU two workgroups.  In us, the three forms and, last, eight tokens at a
  // time with FMA, 2,048 channels in blocks of 256: 64 tokens 16 / 17 / 28 / 26; 100 single tokens 26 / 25 / 37 / 26;
  // 200 29 / 25 / 34 / 33; 500 57 / 29 / 35 / 52; 800 77 / 44 / 48 / 82; 1,500 141 / 67 / 61 / 140; 512 channels in blocks of 128: 100 9.5 /
  // 13 / 17 / 13; 640 14 / 13 / 17 / 17; one block of 1,024: 100 58 / 75 / 110 / 89; 200 108 / 75 / 114 / 94; 1,500 673 / 155 / 220 / 405.
  const int tiles = ceil_div(n, kGateTile), cus = device_cus();
  const long lds = (long)kGateTile * ((ceil_div(bs, 16) * 16 < kGateChunk ? ceil_div(bs, 16) * 16 : kGateChunk) + 4) * 4;
  const int side = 160 * 1024 / lds < 3 ? (int)(160 * 1024 / lds) : 3;
  const bool few = (long)tiles * blocks * ceil_div(bs, kGateTile) <= (long)side * cus;
  const bool many = (long)ceil_div(tiles, 2) * blocks * ceil_div(bs, 8 * kGateTile) >= 2L * cus;
#define KLLM_LRP(NT, KS, OW, TAPS)                                                                                        \
  recurrence_prep_launch<NT, KS, OW, TAPS>(bs, proj, nsplit, split_stride, x_bias, conv_w, conv_b, taps, state, slot_stride, wr_t, \
                                     wi_t, br, bi, rate, span_of_token, slots, span_start, span_pos, a_out, b_out, n, W,  \
                                     blocks, stream)
#define KLLM_LRP_TAPS(TAPS) (few ? KLLM_LRP(1, 4, 1, TAPS) : many ? KLLM_LRP(2, 1, 8, TAPS) : KLLM_LRP(1, 1, 8, TAPS))
  if (taps == 4) return KLLM_LRP_TAPS(4);
  return taps <= 8 ? KLLM_LRP_TAPS(8) : KLLM_LRP_TAPS(0);
#undef KLLM_LRP_TAPS
#undef KLLM_LRP
}

extern "C" int kllm_linear_recurrence_scan(const float* a_in, const float* b_in, const float* proj, int nsplit,
                                           long split_stride, const float* y_bias, float* state, long slot_stride,
                                           const int* slots, const int* span_start, const int* span_pos, void* out,
                                           int n, int n_spans, int longest, int W, int dtype, float* conv_state,
                                           const float* conv_bias, int taps, hipStream_t stream) {
  KLLM_REQUIRE(a_in && b_in && proj && y_bias && state && slots && span_start && span_pos && out,
               "linear_recurrence_scan: null pointer");
  KLLM_REQUIRE(n > 0 && n_spans > 0 && n_spans <= 65535 && W > 0 && nsplit >= 1,
               "linear_recurrence_scan: bad sizes n=%d spans=%d W=%d", n, n_spans, W);
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "linear_recurrence_scan: unknown dtype %d", dtype);
  KLLM_REQUIRE(!conv_state || (taps >= 1 && taps <= kMaxTaps), "linear_recurrence_scan: %d taps (1 to %d)", taps, kMaxTaps);
  const ConvTail tail = {proj, split_stride, 2L * W, conv_bias, conv_state, nsplit, W, W, conv_state ? taps : 0};      // (of x)
#define KLLM_LRS(CH, SEGS)                                                                                               \
  do {                                                                                                                  \
    const bool apart = tail.taps > 1 && (SEGS > 1 || (long)n_spans * ceil_div(W, CH) <= 12L * device_cus());            \
    const dim3 grid(ceil_div(W, CH) + (apart ? ceil_div(W, CH * SEGS) : 0), n_spans), wg(CH * SEGS);                    \
    if (dtype == DT_F32)                                                                                                \
      hipLaunchKernelGGL((linear_recurrence_scan_kernel<float, CH, SEGS>), grid, wg, 0, stream, span_start, slots,      \
                         span_pos, a_in, b_in, proj, W, nsplit, split_stride, y_bias, state, slot_stride, (float*)out, tail);  \
    else                                                                                                                \
      hipLaunchKernelGGL((linear_recurrence_scan_kernel<bf16_t, CH, SEGS>), grid, wg, 0, stream, span_start, slots,     \
                         span_pos, a_in, b_in, proj, W, nsplit, split_stride, y_bias, state, slot_stride, (bf16_t*)out, tail);  \
  } while (0)
  // The longest span's chain bounds the time, and every span, however short, takes workgroups.  Up to 16 tokens there
  // is nothing to cut.  A long chain takes 64 segments of 16 channels where the tokens are those of few
  // long spans (their workgroups of 1,024 threads, one a CU, run at once), else 32 of 32, and below 128 tokens 16 of 32.
  // In us at 2,048 channels, 64 segments of 16 / 32 of 32 / 16 of 32 / 16 of 64 channels:
  //   1,500 tokens 32 / 49 / 85 / 97; 3 x 500 27 / 20 / 32 / 35; 480 beside 4 single tokens 11 / 15 / 19 / 24;
  //   512 beside 60 33 / 23 / 25 / 33; 8 x 250 35 / 23 / 22 / 22; 100 6.2 / 7.0 / 6.6 / 7.6; 40 beside 3 6.1 / 5.7 / 5.7 / 6.4;
  //   16 x 64 28 / 19 / 14 / 15; 8 x 64 13 / 10 / 7.3 / 7.7; 60 x 16 59 / 33 / 22 / 36, uncut 11; 60 x 3 24 / 13 / 9.3 / 15, uncut 4.9.
  // (64 segments of 16 for every step that is not all single tokens, without leaving early: 512 beside 60 66, 60 x 3 56.)
  if (longest <= 0) longest = n > n_spans ? n - n_spans + 1 : 1;      // not said: the most if no span is empty
  const long together = (long)n * ceil_div(W, 16);
  if (longest <= 16) KLLM_LRS(64, 1);
  else if (longest < 128) KLLM_LRS(32, 16);
  else if (together <= (long)device_cus() * longest) KLLM_LRS(16, 64);
  else KLLM_LRS(32, 32);
#undef KLLM_LRS
  KLLM_CHECK_LAUNCH("linear_recurrence_scan");
  return 0;
}
