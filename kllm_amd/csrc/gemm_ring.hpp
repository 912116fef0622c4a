// Products of prompt size (gemm_ring.hip), as gemm.hip's launchers call them.
#pragma once
#include <hip/hip_runtime.h>

namespace kllm {

// What a product's tiles leave: float32 sums [nsplit][n][m], or the storage type (nsplit 1).
enum : int { RING_SUMS = 0, RING_GATE = 1, RING_UNARY = 2 };

// y = x[n][k] . w[m][k]^T, operands float32 (`f32`) or bfloat16: RING_SUMS with `f32_out` or rounded; RING_GATE: w has 2 m rows (gate, up) and
// y = act(gate) * up; RING_UNARY: y = unary_act(sums).  0 or an error.
int gemm_ring(const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int mode, bool f32, bool f32_out,
              int act, const float* act_params, hipStream_t stream);

}  // namespace kllm
