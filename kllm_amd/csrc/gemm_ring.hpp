// Products of prompt size (gemm_ring.hip), as gemm.hip's launchers call them.
#pragma once
#include <hip/hip_runtime.h>

namespace kllm {

// What a product's tiles leave: float32 sums [nsplit][n][m], or the storage type (nsplit 1).
enum : int { RING_SUMS = 0, RING_GATE = 1, RING_UNARY = 2, RING_ROPE = 3 };

// RING_ROPE: w's rows are the queries', keys' and values' heads, H + 2 KV (no cache: H) of 2 half each; queries, rotated, go to y [n][H 2 half], keys
// and values to the pages.
struct RingRope {
  const float* cos_t;      // [n][half], or null: nothing turns
  const float* sin_t;
  void* cache;             // [page][2][KV][page_size 2 half], values [2 half][page_size]; or null
  const int* positions;
  const int* span_of_token;
  const int* block_table;  // [span][max_pages]
  int max_pages, page_size, H, KV, half;      // half: a multiple of 4
};

// y = x[n][k] . w[m][k]^T, operands float32 (`f32`) or bfloat16: RING_SUMS with `f32_out` or rounded; RING_GATE: w has 2 m rows (gate, up) and
// y = act(gate) * up; RING_UNARY: y = unary_act(sums); RING_ROPE: m is half of w's rows, below 2^32 bytes.  0 or an error.
int gemm_ring(const void* x, const void* w, void* y, int n, int m, int k, int nsplit, int mode, bool f32, bool f32_out,
              int act, const float* act_params, hipStream_t stream, const RingRope& rope = RingRope());

}  // namespace kllm
