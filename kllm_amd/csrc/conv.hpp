// A short causal convolution per channel: y_t = sum_j w[c][j] x_(t - taps + 1 + j), zeros before
// position 0, over inputs that arrive as float32 sums [nsplit][n][cols] of a step's projections.
// The inputs of the last taps - 1 positions are part of a request's state ([C][taps - 1] per
// slot, oldest first); the first tokens of a span read them there.
#pragma once

#include "common.hpp"

namespace kllm {

constexpr int kMaxTaps = 16;

// The input of the convolution at row `row` of the step (a token of the same span), channel c.
__device__ __forceinline__ float conv_input(const float* __restrict__ proj, int nsplit, long split_stride, long cols,
                                            long col, const float* __restrict__ bias, long row) {
  const float* p = proj + row * cols + col;
  float v = 0.f;
  for (int s = 0; s < nsplit; ++s) v += p[s * split_stride];
  return bias ? v + bias[col] : v;
}

// The convolution's output for the token at row t (span rows from t0, `fresh`: the span starts at
// position 0), channel c of C, whose input column is col0 + c; `st` is the request's
// [C][taps - 1] entries.
__device__ __forceinline__ float conv_at(const float* __restrict__ proj, int nsplit, long split_stride, long cols,
                                         long col, const float* __restrict__ in_bias,
                                         const float* __restrict__ w_row, int taps, const float* __restrict__ st_row,
                                         bool fresh, long t, long t0) {
  float y = 0.f;
  const int K = taps - 1;
  for (int j = 0; j < taps; ++j) {
    const long row = t - K + j;
    float x;
    if (row >= t0) x = conv_input(proj, nsplit, split_stride, cols, col, in_bias, row);
    else x = fresh ? 0.f : st_row[K - (int)(t0 - row)];
    y = fmaf(w_row[j], x, y);
  }
  return y;
}

// What a step leaves of a convolution's inputs: the entries of a request's state take those of the span's last
// taps - 1 positions; where the span is shorter, the entries it had move up (zeros where it starts at position 0).
// Work of a launch behind the one that reads the entries; taps 0: nothing to do.
struct ConvTail {
  const float* proj;        // [nsplit][n][cols], the inputs in columns col0 .. col0 + C
  long split_stride, cols;
  const float* in_bias;     // [C], or null
  float* state;             // the field's place in the first slot
  int nsplit, col0, C, taps;
};

__device__ __forceinline__ void conv_tail(const ConvTail& v, long slot_stride, int c, int slot, long t0, long t1, bool fresh) {
  const int K = v.taps - 1;
  float* st = v.state + (long)slot * slot_stride + (long)c * K;
  const float* bias = v.in_bias ? v.in_bias - v.col0 : nullptr;
  const int len = (int)min(t1 - t0, (long)K);
  auto input = [&](long row) { return conv_input(v.proj, v.nsplit, v.split_stride, v.cols, v.col0 + c, bias, row); };
  if (v.taps == 4) {                     // every load asked for at once
    float old[3], in[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      old[j] = st[j];
      in[j] = len > 0 ? input(t1 - min(3 - j, len)) : 0.f;        // (a row that is there; used where it is the right one)
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const float kept = len == 0 ? old[j] : len == 1 ? old[j < 2 ? j + 1 : j] : old[2];
      st[j] = j + len >= 3 ? in[j] : fresh ? 0.f : kept;
    }
  } else {
    for (int j = 0; j < K; ++j)          // (an entry that moves up is read before it is written)
      st[j] = j + len >= K ? input(t1 - K + j) : fresh ? 0.f : st[j + len];
  }
}

}  // namespace kllm
