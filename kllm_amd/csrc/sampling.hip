// Choosing the next token on the device, one workgroup per row of logits.
//
// temperature == 0: the largest logit, the first one on ties (the reference's
// host Argmax, engine/engine.go:216-224).  temperature > 0:
// p = softmax(logits / temperature) with the maximum subtracted, all in
// 32-bit, and the smallest index whose cumulative probability exceeds
// u * total, for a uniform u in [0, 1) that the caller draws.
#include <math.h>

#include <type_traits>

#include "common.hpp"
#include "kllm_kernels.h"

namespace kllm {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / kWave;

// One workgroup a row: a row's logits come in one trip (up to 32,768; 128,256 in four), and what follows is a chain of lane exchanges, so
// the maximum goes by data-parallel moves and its place by asking the lanes that have it: 8 rows of 32,000 8.9 -> 5.7 us (contiguous segments a
// thread and twelve exchanges through LDS a wave before).
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(
    int* __restrict__ out, const float* __restrict__ logits, const float* __restrict__ temperature,
    const float* __restrict__ uniform, int vocab) {
  __shared__ float wave_val[kSampleWaves];
  __shared__ int wave_idx[kSampleWaves];
  __shared__ float wave_tot[kSampleWaves];
  __shared__ int chosen;

  const int r = blockIdx.x, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const float* row = logits + (long)r * vocab;
  // (asked for here, so that the trip to memory runs beside the logits')
  const float temp = temperature ? temperature[r] : 0.f;
  const float u = uniform ? uniform[r] : 0.f;
  // For the sums, and the maximum of a row in no whole pieces, each thread owns one contiguous segment, so thread order is index order.
  const int seg = (vocab + 4 * kSampleThreads - 1) / (4 * kSampleThreads) * 4;
  const int lo = min(tid * seg, vocab), hi = min(lo + seg, vocab);

  // The greatest logit and the first place that has it (numbers only: a NaN is never chosen before one that is none).
  float bv = -INFINITY, wm;
  int bi = vocab;  // "none": loses against every index
  if (vocab % 4 == 0 && ((uintptr_t)logits & 15) == 0) {
    // pieces of 16 bytes, neighbouring threads side by side, eight of them in flight a thread; a wave looks a turn through where
    // a lane has more than the wave's greatest so far (of 256,000 logits 28.0 -> 20.1 us), and no pieces that are not there (of 1,000 5.0 -> 3.0)
    const int pieces = vocab / 4;
    wm = -INFINITY;
    auto turn = [&](int first, auto whole) {
      constexpr bool WHOLE = decltype(whole)::value;
      const int p0 = first + tid;
      floatx4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (!WHOLE) v[j] = floatx4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (WHOLE || first + j * kSampleThreads < pieces)
          v[j] = *reinterpret_cast<const floatx4*>(row + 4 * min(p0 + j * kSampleThreads, pieces - 1));
      }
      if (wm != -INFINITY) {
        float most = v[0][0];
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) most = fmaxf(most, v[j][e]);
        if (!__builtin_amdgcn_ballot_w64(most > wm)) return;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (!WHOLE && first + j * kSampleThreads >= pieces) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * (p0 + j * kSampleThreads) + e;
          if (i < vocab && (v[j][e] > bv || (bi == vocab && v[j][e] == bv))) { bv = v[j][e]; bi = i; }   // strict: the first maximum stays
        }
      }
      wm = wave_max(bv);
    };
    for (int first = 0; first < pieces; first += 8 * kSampleThreads) {
      if (pieces - first > 7 * kSampleThreads) turn(first, std::true_type()); else turn(first, std::false_type());
    }
  } else {
    for (int i = lo; i < hi; ++i) {
      const float v = row[i];
      if (v > bv || (bi == vocab && v == bv)) { bv = v; bi = i; }
    }
    wm = wave_max(bv);
  }
  // The lanes that have the greatest, mostly one, are asked for their places.
  auto first_of = [&](float v, int i, float greatest) {
    int best = vocab;
    for (unsigned long m = __builtin_amdgcn_ballot_w64(v == greatest && i < vocab); m; m &= m - 1)     // (a lane without a number has no place)
      best = min(best, __builtin_amdgcn_readlane(i, __builtin_ctzl(m)));
    return best;
  };
  const int wi = first_of(bv, bi, wm);
  if (lane == 0) {
    wave_val[wave] = wm;
    wave_idx[wave] = wi;
  }
  if (tid == 0) chosen = vocab - 1;
  __syncthreads();
  const float wv = wave_val[lane % kSampleWaves];
  const float mx = wave_max(wv);
  int arg = first_of(wv, wave_idx[lane % kSampleWaves], mx);
  if (arg == vocab) arg = 0;      // nothing but NaN
  if (!(temp > 0.f)) {
    if (tid == 0) out[r] = arg;
    return;
  }
  const float inv_t = 1.f / temp;
  float sum = 0.f;
  for (int i = lo; i < hi; ++i) sum += expf((row[i] - mx) * inv_t);
  // inclusive scan over the wave, then over the waves: thread t's probability
  // mass lies in [incl - sum, incl)
  float incl = sum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const float up = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += up;
  }
  if (lane == kWave - 1) wave_tot[wave] = incl;
  __syncthreads();
  float before = 0.f, total = 0.f;
  for (int w = 0; w < kSampleWaves; ++w) {
    if (w < wave) before += wave_tot[w];
    total += wave_tot[w];
  }
  // excl is the previous thread's incl, bit for bit: the ranges leave no gap
  const float prev = __shfl_up(incl, 1, kWave);
  const float excl = before + (lane == 0 ? 0.f : prev);
  incl += before;
  const float target = u * total;
  if (sum > 0.f && target >= excl && target < incl) {
    float c = excl;
    int idx = hi - 1;
    for (int i = lo; i < hi; ++i) {
      c += expf((row[i] - mx) * inv_t);
      if (target < c) { idx = i; break; }
    }
    chosen = idx;
  }
  __syncthreads();
  if (tid == 0) out[r] = chosen;
}

}  // namespace kllm

using namespace kllm;

extern "C" int kllm_sample(int* out, const float* logits, const float* temperature,
                           const float* uniform, int rows, int vocab, hipStream_t stream) {
  KLLM_REQUIRE(out && logits, "sample: null pointer");
  KLLM_REQUIRE(rows > 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", rows, vocab);
  KLLM_REQUIRE((temperature == nullptr) == (uniform == nullptr),
               "sample: temperatures and uniforms go together");
  hipLaunchKernelGGL(sample_kernel, dim3(rows), dim3(kSampleThreads), 0, stream, out, logits,
                     temperature, uniform, vocab);
  KLLM_CHECK_LAUNCH("sample");
  return 0;
}
