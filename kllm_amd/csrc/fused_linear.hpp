// What the decode-batch products (fused_linear.hip) and the products of up to 64 rows without staging
// (linear_rows.hip) share: the output's description, its kinds and the rotation's stores.
#pragma once

#include "common.hpp"

namespace kllm {

constexpr int FL_SS_LOADS = 4;     // 16-byte loads per lane of a row's partial sums of squares: 16 lanes a row
constexpr int FL_SS_MAX = 16 * 4 * FL_SS_LOADS;   // partial sums of squares per row at most

enum : int { FL_PARTS = 0, FL_RESID = 1, FL_SWIGLU = 2, FL_ROPE = 3 };
// FL_PARTS with act >= FL_UNARY: y is [n][m] in the storage type = unary_act(sums, act - FL_UNARY), the
// activation's learned constants (if it has any) behind norm_w.
constexpr int FL_UNARY = 16;

struct FlOut {
  void* y;
  const float* cos_t;
  const float* sin_t;
  void* cache;
  const int* positions;
  const int* span_of_token;
  const int* block_table;
  int max_pages, page_size, H, KV, hd;
  int act;                      // the gate's activation (FL_SWIGLU)
  float* resid;                 // FL_RESID: the residual stream [n][m]; y receives resid * norm_w in the storage type
  const float* norm_w;          // FL_RESID: weight [m] of the norm behind the addition
  float* ss_out;                // FL_RESID: [n][workgroups rounded up to 4] sums of squares of the new rows
  const float* ss_in;           // SCALED: [n][ss_parts rounded up to 4], what a FL_RESID product left
  int ss_parts;
  float eps;
  int tiled;                    // W is the copy that fl_tile_kernel made for this epilogue (see there)
  int x_tiled, y_tiled;         // linear_rows: rows in the lanes' order
};

// Row of W behind MFMA row c of a tile, or -1.  Pair epilogues: unit = pair.
template <int EP>
__device__ __forceinline__ long fl_row(int tile, int c, int m, const FlOut& o) {
  if (EP == FL_PARTS || EP == FL_RESID) {
    const long r = (long)tile * 16 + c;
    return r < m ? r : -1;
  }
  const int pair = tile * 8 + (c & 7);          // m < 2^31, so pairs and tiles fit an int
  const int pairs = m / 2;
  if (pair >= pairs) return -1;
  const bool second = c >= 8;
  if (EP == FL_SWIGLU) return second ? pairs + pair : pair;
  const int half = o.hd / 2;
  const int rot_pairs = (o.H + (o.cache ? o.KV : 0)) * half;
  if (pair < rot_pairs) {
    const long a = (long)(pair / half) * o.hd + pair % half;   // q and k rows follow each other in W
    return second ? a + half : a;
  }
  const long e = 2 * (long)(pair - rot_pairs);
  return (long)(o.H + o.KV) * o.hd + e + (second ? 1 : 0);
}

// A workgroup barrier for data in LDS.  Unlike __syncthreads it does not wait for loads from
// memory: the weights asked for ahead stay in flight while the waves meet.
__device__ __forceinline__ void fl_lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0): this wave's LDS operations are done
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Pair `pair` (sums a and b) of row xr of a rotation product: a query's or key's elements j and j + hd/2,
// rotated, or two neighbouring elements of a value.
template <typename T>
__device__ __forceinline__ void fl_rope_store(const FlOut& out, int xr, int pair, float a, float b, float cc, float sn,
                                              int page, int slot) {
  const int half = out.hd / 2;
  const int q_pairs = out.H * half, k_pairs = out.cache ? out.KV * half : 0;
  const int region = pair < q_pairs ? 0 : pair < q_pairs + k_pairs ? 1 : 2;
  const long block = (long)out.page_size * out.hd;
  if (region < 2) {
    const int p = region ? pair - q_pairs : pair;
    const int head = p / half, j = p % half;
    const float ra = a * cc - b * sn, rb = b * cc + a * sn;
    T* o = region == 0 ? reinterpret_cast<T*>(out.y) + ((long)xr * out.H + head) * out.hd
                       : reinterpret_cast<T*>(out.cache) + (((long)page * 2 + 0) * out.KV + head) * block + (long)slot * out.hd;
    o[j] = from_f32<T>(ra);
    o[j + half] = from_f32<T>(rb);
  } else {
    const int e = 2 * (pair - q_pairs - k_pairs);
    const int head = e / out.hd, j = e % out.hd;
    T* v = reinterpret_cast<T*>(out.cache) + (((long)page * 2 + 1) * out.KV + head) * block;
    v[(long)j * out.page_size + slot] = from_f32<T>(a);
    v[(long)(j + 1) * out.page_size + slot] = from_f32<T>(b);
  }
}

}  // namespace kllm
