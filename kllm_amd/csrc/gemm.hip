// Matrix products Y[n, m] = X[n, k] . W[m, k]^T (weights are [out, in], as the
// reference keeps them: backend/model.cu:494-503).  Accumulation is always in
// 32-bit.  Five kernels:
//
//   plain   one thread per output; any size; the yardstick the others are
//           tested against
//   tiled   true 32-bit FMA tiles through LDS, for the float32 engine
//   mfma    MFMA tiles through LDS (gemm_ring.hip), both types; float32 with 32-bit operands, products
//           and sums: no reduced precision
//   skinny  bfloat16 MFMA 16x16x32, weights streamed straight from memory,
//           for up to 64 rows of X (decode batches); K may be split
//   gemv    one wave per weight row, up to 8 rows of X; K may be split
//
// A split product writes `nsplit` partial results [nsplit][n][m] in float32;
// the consumer adds them.
#include "common.hpp"
#include "gemm_ring.hpp"
#include "kllm_kernels.h"

namespace kllm {

// ------------------------------------------------------------------ plain
template <typename T, typename TOUT>
__global__ void gemm_plain_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                  TOUT* __restrict__ Y, int n, int m, int k) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)n * m) return;
  const int r = idx / m, c = idx % m;
  const T* x = X + (long)r * k;
  const T* w = W + (long)c * k;
  float acc = 0.f;
  for (int i = 0; i < k; ++i) acc = fmaf(to_f32(x[i]), to_f32(w[i]), acc);
  Y[idx] = from_f32<TOUT>(acc);
}

// ------------------------------------------------------------------ tiled f32
constexpr int TBM = 64, TBN = 64, TBK = 16;

template <typename TOUT>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ X,
                                                             const float* __restrict__ W,
                                                             TOUT* __restrict__ Y, int n, int m,
                                                             int k, int vec_ok) {
  __shared__ float Xs[TBK][TBM + 4];
  __shared__ float Ws[TBK][TBN + 4];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const long row0 = (long)blockIdx.y * TBM, col0 = (long)blockIdx.x * TBN;
  const int lr = tid / 4, lk = (tid % 4) * 4;  // this thread's part of a tile load

  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < k; k0 += TBK) {
    float xv[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {0.f, 0.f, 0.f, 0.f};
    const long xr = row0 + lr, wr = col0 + lr;
    const int kk = k0 + lk;
    if (xr < n) {
      const float* p = X + xr * k + kk;
      if (vec_ok && kk + 3 < k) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        xv[0] = v.x; xv[1] = v.y; xv[2] = v.z; xv[3] = v.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) if (kk + i < k) xv[i] = p[i];
      }
    }
    if (wr < m) {
      const float* p = W + wr * k + kk;
      if (vec_ok && kk + 3 < k) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        wv[0] = v.x; wv[1] = v.y; wv[2] = v.z; wv[3] = v.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) if (kk + i < k) wv[i] = p[i];
      }
    }
    __syncthreads();  // the previous tile is no longer read
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      Xs[lk + i][lr] = xv[i];
      Ws[lk + i][lr] = wv[i];
    }
    __syncthreads();
#pragma unroll
    for (int kk2 = 0; kk2 < TBK; ++kk2) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = Xs[kk2][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Ws[kk2][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long r = row0 + ty * 4 + i;
    if (r >= n) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const long c = col0 + tx * 4 + j;
      if (c < m) Y[r * m + c] = from_f32<TOUT>(acc[i][j]);
    }
  }
}

// ------------------------------------------------------------------ bf16 MFMA skinny
// Up to 16*NT rows of X (decode batches).  A workgroup takes 64 rows of W and
// one slice of K: it first puts its slice of X into LDS, then each of its four
// waves streams 16 rows of W straight from memory, eight 16-byte loads ahead,
// and multiplies them with X from LDS.  MFMA 16x16x32 with A = W tile,
// B = X^T, so D[w row][x row]: lane l (g = l/16, c = l%16) holds
// A[c][8g..8g+7], B[8g..8g+7][c], D[4g+i][c].
constexpr int SK_SLICE_MAX = 512;             // K per workgroup at most
constexpr int SK_LD = SK_SLICE_MAX + 8;       // LDS row stride (elements): 16-byte reads conflict-free
constexpr int SK_AHEAD = 8;                   // W loads in flight per lane

template <int NT, int RT>   // NT: 16-row tiles of X; RT: 16-row tiles of W per wave (1 or 2)
__global__ __launch_bounds__(256) void gemm_bf16_skinny_kernel(const bf16_t* __restrict__ X,
                                                               const bf16_t* __restrict__ W,
                                                               float* __restrict__ Y, int n, int m,
                                                               int k, int kslice) {
  extern __shared__ __attribute__((aligned(16))) bf16_t xs[];   // [NT*16][SK_LD]
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int g = lane / 16, c = lane % 16;
  const int kbeg = blockIdx.y * kslice;
  const int kend = min(k, kbeg + kslice);
  const int klen = kend - kbeg;                                  // a multiple of 8
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};

  // This wave's rows of W; their first loads go out before X is staged.  With RT = 2 a
  // wave multiplies every piece of X it reads from LDS with two tiles of W, and a
  // workgroup stages X once for 128 rows of W instead of 64.
  const long m0 = ((long)blockIdx.x * 4 + wave) * 16 * RT;
  const bf16_t* wp[RT];
  bool wok[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const long wrow = m0 + rt * 16 + c;
    wok[rt] = wrow < m;
    wp[rt] = W + (wok[rt] ? wrow : 0) * k + kbeg + 8 * g;
  }
  const int steps = (klen + 31) / 32;
  auto load_a = [&](int rt, int s) -> bf16x8 {
    return (wok[rt] && s < steps && 32 * s + 8 * g < klen) ? *reinterpret_cast<const bf16x8*>(wp[rt] + 32 * s)
                                                            : zero;
  };
  bf16x8 cur[RT][SK_AHEAD], nxt[RT][SK_AHEAD];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int u = 0; u < SK_AHEAD; ++u) cur[rt][u] = load_a(rt, u);

  // Stage X[0..16*NT)[kbeg..kend) in LDS, eight 16-byte loads in flight per thread.
  const int chunks = (klen + 7) / 8;
  const int total = NT * 16 * chunks;
  for (int base = tid; base < total; base += 256 * 8) {
    bf16x8 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int idx = base + j * 256;
      const int r = idx / chunks, ch = idx % chunks;
      v[j] = (idx < total && r < n) ? *reinterpret_cast<const bf16x8*>(X + (long)r * k + kbeg + ch * 8) : zero;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int idx = base + j * 256;
      if (idx < total) {
        const int r = idx / chunks, ch = idx % chunks;
        *reinterpret_cast<bf16x8*>(&xs[r * SK_LD + ch * 8]) = v[j];
      }
    }
  }
  __syncthreads();
  if (m0 >= m) return;

  floatx4 acc[RT][NT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[rt][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  for (int s0 = 0; s0 < steps; s0 += SK_AHEAD) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < SK_AHEAD; ++u) nxt[rt][u] = load_a(rt, s0 + SK_AHEAD + u);
#pragma unroll
    for (int u = 0; u < SK_AHEAD; ++u) {
      const int s1 = s0 + u;
      if (s1 < steps) {
        const bool kin = 32 * s1 + 8 * g < klen;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const bf16x8 b = kin ? *reinterpret_cast<const bf16x8*>(&xs[(t * 16 + c) * SK_LD + 32 * s1 + 8 * g])
                               : zero;
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[rt][u], b, acc[rt][t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int u = 0; u < SK_AHEAD; ++u) cur[rt][u] = nxt[rt][u];
  }

  // A lane holds four neighbouring columns of one row of X: one 16-byte store where the
  // row length allows it.
  float* out = Y + (long)blockIdx.y * n * m;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const long col0 = m0 + rt * 16 + 4 * g;
    const bool vec = m % 4 == 0 && col0 + 3 < m && ((uintptr_t)Y & 15) == 0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int xr = t * 16 + c;
      if (xr >= n) continue;
      if (vec) {
        *reinterpret_cast<floatx4*>(&out[(long)xr * m + col0]) = acc[rt][t];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (col0 + i < m) out[(long)xr * m + col0 + i] = acc[rt][t][i];
      }
    }
  }
}

// ------------------------------------------------------------------ gemv
// One wave per row of W, NT (<= 8) rows of X; lanes stride over K in chunks
// of 8 elements.  Four rows of W per workgroup.
template <typename T, int NT>
__global__ __launch_bounds__(256) void gemv_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                   float* __restrict__ Y, int n, int m, int k,
                                                   int kslice, int vec_ok) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const long row = (long)blockIdx.x * 4 + wave;
  if (row >= m) return;
  const int kbeg = blockIdx.y * kslice;
  const int kend = min(k, kbeg + kslice);
  const T* w = W + row * k;
  float acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = 0.f;

  constexpr int V = 16 / sizeof(T);  // elements per 16-byte load
  typedef T vec_t __attribute__((ext_vector_type(V)));
  if (vec_ok) {
    for (int i = kbeg + lane * V; i < kend; i += kWave * V) {
      const vec_t wv = *reinterpret_cast<const vec_t*>(w + i);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (t < n) {
          const vec_t xv = *reinterpret_cast<const vec_t*>(X + (long)t * k + i);
#pragma unroll
          for (int e = 0; e < V; ++e) acc[t] = fmaf(to_f32(wv[e]), to_f32(xv[e]), acc[t]);
        }
      }
    }
  } else {
    for (int i = kbeg + lane; i < kend; i += kWave) {
      const float wv = to_f32(w[i]);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < n) acc[t] = fmaf(wv, to_f32(X[(long)t * k + i]), acc[t]);
    }
  }
  float* out = Y + (long)blockIdx.y * n * m;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const float s = wave_sum(acc[t]);
    if (lane == 0 && t < n) out[(long)t * m + row] = s;
  }
}

// ------------------------------------------------------------------ streaming gemv
// Up to 4 rows of X.  A wave takes R rows of W and one slice of K and has all
// of a slice's loads in flight at once: U steps of 64 lanes x 16 bytes per row.
template <typename T, int NT, int R, int U>
__global__ __launch_bounds__(256) void gemv_stream_kernel(const T* __restrict__ X,
                                                          const T* __restrict__ W,
                                                          float* __restrict__ Y, int n, int m, int k,
                                                          int kslice) {
  constexpr int V = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const long row0 = ((long)blockIdx.x * 4 + wave) * R;
  if (row0 >= m) return;
  const int kbeg = blockIdx.y * kslice;
  const int kend = min(k, kbeg + kslice);
  float acc[R][NT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[r][t] = 0.f;

  for (int k0 = kbeg + lane * V; k0 < kend; k0 += U * kWave * V) {
    vec_t wv[U][R], xv[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k0 + u * kWave * V;
      const bool kin = kk < kend;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool ok = kin && row0 + r < m;
        wv[u][r] = ok ? *reinterpret_cast<const vec_t*>(W + (row0 + r) * k + kk) : vec_t{};
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bool ok = kin && t < n;
        xv[u][t] = ok ? *reinterpret_cast<const vec_t*>(X + (long)t * k + kk) : vec_t{};
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < V; ++e)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float wf = to_f32(wv[u][r][e]);
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[r][t] = fmaf(wf, to_f32(xv[u][t][e]), acc[r][t]);
        }
  }
  float* out = Y + (long)blockIdx.y * n * m;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float sum = wave_sum(acc[r][t]);
      if (lane == 0 && t < n && row0 + r < m) out[(long)t * m + row0 + r] = sum;
    }
}

}  // namespace kllm

using namespace kllm;

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The 64-row variant of the skinny kernel stages 66,560 bytes of LDS, above the
// default limit of a launch; raise it once per kernel.
template <int NT, int RT>
static int launch_skinny(const bf16_t* x, const bf16_t* w, float* y, int n, int m, int k, int kslice,
                         int nsplit, hipStream_t stream) {
  static int raised = 0;
  const size_t lds = (size_t)NT * 16 * SK_LD * sizeof(bf16_t);
  if (!raised) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_bf16_skinny_kernel<NT, RT>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) KLLM_FAIL((int)e, "gemm skinny: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = 1;
  }
  const dim3 grid(ceil_div(m, 64 * RT), nsplit);
  hipLaunchKernelGGL((gemm_bf16_skinny_kernel<NT, RT>), grid, dim3(256), lds, stream, x, w, y, n, m, k, kslice);
  return 0;
}

extern "C" int kllm_gemm(const void* x, const void* w, void* y, int n, int m, int k, int dtype,
                         int out_dtype, int algo, int nsplit, hipStream_t stream) {
  KLLM_REQUIRE(x && w && y, "gemm: null pointer");
  KLLM_REQUIRE(n > 0 && m > 0 && k > 0, "gemm: bad sizes n=%d m=%d k=%d", n, m, k);
  KLLM_REQUIRE(dtype == DT_F32 || dtype == DT_BF16, "gemm: unknown dtype %d", dtype);
  KLLM_REQUIRE(out_dtype == DT_F32 || out_dtype == dtype, "gemm: output dtype %d with input %d",
               out_dtype, dtype);
  KLLM_REQUIRE(nsplit >= 1 && nsplit <= 256, "gemm: nsplit %d is outside [1, 256]", nsplit);
  KLLM_REQUIRE((long)n * m < (1L << 31) && (long)m * k < (1L << 40), "gemm: sizes overflow");

  if (algo == KLLM_GEMM_PLAIN) {
    KLLM_REQUIRE(nsplit == 1, "gemm plain: no split");
    const long total = (long)n * m;
    const dim3 grid(ceil_div(total, 256));
    if (dtype == DT_F32)
      hipLaunchKernelGGL((gemm_plain_kernel<float, float>), grid, dim3(256), 0, stream,
                         (const float*)x, (const float*)w, (float*)y, n, m, k);
    else if (out_dtype == DT_F32)
      hipLaunchKernelGGL((gemm_plain_kernel<bf16_t, float>), grid, dim3(256), 0, stream,
                         (const bf16_t*)x, (const bf16_t*)w, (float*)y, n, m, k);
    else
      hipLaunchKernelGGL((gemm_plain_kernel<bf16_t, bf16_t>), grid, dim3(256), 0, stream,
                         (const bf16_t*)x, (const bf16_t*)w, (bf16_t*)y, n, m, k);
    KLLM_CHECK_LAUNCH("gemm plain");
    return 0;
  }

  if (algo == KLLM_GEMM_TILED_F32) {
    KLLM_REQUIRE(dtype == DT_F32 && out_dtype == DT_F32, "gemm tiled: float32 only");
    KLLM_REQUIRE(nsplit == 1, "gemm tiled: no split");
    const int vec_ok = (k % 4 == 0) && aligned16(x) && aligned16(w);
    const dim3 grid(ceil_div(m, TBN), ceil_div(n, TBM));
    hipLaunchKernelGGL((gemm_f32_tiled_kernel<float>), grid, dim3(256), 0, stream, (const float*)x,
                       (const float*)w, (float*)y, n, m, k, vec_ok);
    KLLM_CHECK_LAUNCH("gemm tiled");
    return 0;
  }

  if (algo == KLLM_GEMM_MFMA_BF16 || algo == KLLM_GEMM_MFMA_F32) {
    const bool f32 = algo == KLLM_GEMM_MFMA_F32;
    const int stage = f32 ? 32 : 64, chunk = f32 ? 4 : 8;   // elements of K per stage, per 16 bytes
    KLLM_REQUIRE(dtype == (f32 ? DT_F32 : DT_BF16), "gemm mfma: algorithm %d does not take dtype %d", algo, dtype);
    KLLM_REQUIRE(nsplit == 1 || out_dtype == DT_F32, "gemm mfma: K is split only for float32 partial sums");
    KLLM_REQUIRE(nsplit <= 16 && (long)(ceil_div(ceil_div(k, nsplit), stage) * stage) * (nsplit - 1) < k,
                 "gemm mfma: nsplit %d leaves an empty slice of K=%d", nsplit, k);
    KLLM_REQUIRE(k % chunk == 0 && aligned16(x) && aligned16(w),
                 "gemm mfma: K=%d must be a multiple of %d and the operands 16-byte aligned", k, chunk);
    int rc = gemm_ring(x, w, y, n, m, k, out_dtype == DT_F32 ? nsplit : 1, RING_SUMS, f32, out_dtype == DT_F32, -1, nullptr, stream);
    if (rc) return rc;
    KLLM_CHECK_LAUNCH("gemm mfma");
    return 0;
  }

  if (algo == KLLM_GEMM_SKINNY_BF16) {
    KLLM_REQUIRE(dtype == DT_BF16 && out_dtype == DT_F32,
                 "gemm skinny: bfloat16 in, float32 partial sums out");
    KLLM_REQUIRE(n <= 64, "gemm skinny: n=%d exceeds 64", n);
    KLLM_REQUIRE(k % 8 == 0 && aligned16(x) && aligned16(w),
                 "gemm skinny: K=%d must be a multiple of 8 and the operands 16-byte aligned", k);
    const int kslice = ceil_div(ceil_div(k, nsplit), 32) * 32;
    KLLM_REQUIRE(kslice <= SK_SLICE_MAX, "gemm skinny: K=%d in %d slices exceeds %d per slice", k,
                 nsplit, SK_SLICE_MAX);
    KLLM_REQUIRE((long)kslice * (nsplit - 1) < k, "gemm skinny: nsplit %d leaves an empty slice of K=%d",
                 nsplit, k);
    const bf16_t *xp = (const bf16_t*)x, *wp = (const bf16_t*)w;
    float* yp = (float*)y;
    const int nt = ceil_div(n, 16);
    // Many rows of X and of W: two tiles of W per wave, while that still leaves a workgroup
    // for every CU (measured: a gain from 33 rows of X on, a loss below).
    const bool wide = nt >= 3 && (long)ceil_div(m, 128) * nsplit >= 256;
    int rc;
    if (nt == 1) rc = launch_skinny<1, 1>(xp, wp, yp, n, m, k, kslice, nsplit, stream);
    else if (nt == 2) rc = launch_skinny<2, 1>(xp, wp, yp, n, m, k, kslice, nsplit, stream);
    else if (nt == 3) rc = wide ? launch_skinny<3, 2>(xp, wp, yp, n, m, k, kslice, nsplit, stream)
                                : launch_skinny<3, 1>(xp, wp, yp, n, m, k, kslice, nsplit, stream);
    else rc = wide ? launch_skinny<4, 2>(xp, wp, yp, n, m, k, kslice, nsplit, stream)
                   : launch_skinny<4, 1>(xp, wp, yp, n, m, k, kslice, nsplit, stream);
    if (rc) return rc;
    KLLM_CHECK_LAUNCH("gemm skinny");
    return 0;
  }

  if (algo == KLLM_GEMM_GEMV) {
    KLLM_REQUIRE(out_dtype == DT_F32, "gemv: float32 partial sums out");
    KLLM_REQUIRE(n <= 8, "gemv: n=%d exceeds 8", n);
    const int vlen = dtype == DT_F32 ? 4 : 8;
    const int vec_ok = (k % vlen == 0) && aligned16(x) && aligned16(w);
    const int unit = kWave * vlen;
    if (vec_ok && n <= 4) {
      constexpr int R = 2, U = 4;
      const int ks = ceil_div(ceil_div(k, nsplit), unit) * unit;
      KLLM_REQUIRE((long)ks * (nsplit - 1) < k, "gemv: nsplit %d leaves an empty slice of K=%d", nsplit, k);
      const dim3 sgrid(ceil_div(m, 4 * R), nsplit);
#define KLLM_GS(T, NT)                                                                           \
  hipLaunchKernelGGL((gemv_stream_kernel<T, NT, R, U>), sgrid, dim3(256), 0, stream, (const T*)x, \
                     (const T*)w, (float*)y, n, m, k, ks)
      if (dtype == DT_F32) {
        if (n == 1) KLLM_GS(float, 1);
        else if (n == 2) KLLM_GS(float, 2);
        else KLLM_GS(float, 4);
      } else {
        if (n == 1) KLLM_GS(bf16_t, 1);
        else if (n == 2) KLLM_GS(bf16_t, 2);
        else KLLM_GS(bf16_t, 4);
      }
#undef KLLM_GS
      KLLM_CHECK_LAUNCH("gemv stream");
      return 0;
    }
    int kslice = ceil_div(ceil_div(k, nsplit), unit) * unit;
    KLLM_REQUIRE((long)kslice * (nsplit - 1) < k, "gemv: nsplit %d leaves an empty slice of K=%d",
                 nsplit, k);
    const dim3 grid(ceil_div(m, 4), nsplit);
#define KLLM_GEMV(T, NT)                                                                        \
  hipLaunchKernelGGL((gemv_kernel<T, NT>), grid, dim3(256), 0, stream, (const T*)x, (const T*)w, \
                     (float*)y, n, m, k, kslice, vec_ok)
    if (dtype == DT_F32) {
      if (n == 1) KLLM_GEMV(float, 1);
      else if (n == 2) KLLM_GEMV(float, 2);
      else if (n <= 4) KLLM_GEMV(float, 4);
      else KLLM_GEMV(float, 8);
    } else {
      if (n == 1) KLLM_GEMV(bf16_t, 1);
      else if (n == 2) KLLM_GEMV(bf16_t, 2);
      else if (n <= 4) KLLM_GEMV(bf16_t, 4);
      else KLLM_GEMV(bf16_t, 8);
    }
#undef KLLM_GEMV
    KLLM_CHECK_LAUNCH("gemv");
    return 0;
  }
  KLLM_FAIL(ERR_ARG, "gemm: unknown algorithm %d", algo);
}

extern "C" int kllm_gemm_swiglu(const void* x, const void* w_gate_up, void* h, int n, int f, int k,
                                int dtype, int act, hipStream_t stream) {
  KLLM_REQUIRE(x && w_gate_up && h, "gemm_swiglu: null pointer");
  KLLM_REQUIRE(act >= 0 && act < ACT_COUNT, "gemm_swiglu: unknown activation %d", act);
  KLLM_REQUIRE(n > 0 && f > 0 && k > 0, "gemm_swiglu: bad sizes n=%d f=%d k=%d", n, f, k);
  KLLM_REQUIRE(dtype == DT_BF16 || dtype == DT_F32, "gemm_swiglu: unknown dtype %d", dtype);
  const int chunk = dtype == DT_F32 ? 4 : 8;
  KLLM_REQUIRE(k % chunk == 0 && aligned16(x) && aligned16(w_gate_up),
               "gemm_swiglu: K=%d must be a multiple of %d and the operands 16-byte aligned", k, chunk);
  KLLM_REQUIRE((long)n * f < (1L << 31), "gemm_swiglu: sizes overflow");
  if (int rc = gemm_ring(x, w_gate_up, h, n, f, k, 1, RING_GATE, dtype == DT_F32, dtype == DT_F32, act, nullptr, stream)) return rc;
  KLLM_CHECK_LAUNCH("gemm_swiglu");
  return 0;
}

// h[n][m] = act(x . w^T) in dtype, the activation (one without a gate) in the product's epilogue.
extern "C" int kllm_gemm_act(const void* x, const void* w, void* h, int n, int m, int k, int dtype, int act,
                             const float* act_params, hipStream_t stream) {
  KLLM_REQUIRE(x && w && h, "gemm_act: null pointer");
  KLLM_REQUIRE(act >= 0 && act < UNARY_ACT_COUNT, "gemm_act: unknown activation %d", act);
  KLLM_REQUIRE(act != ACT_XIELU || act_params, "gemm_act: this activation needs its two constants");
  KLLM_REQUIRE(n > 0 && m > 0 && k > 0, "gemm_act: bad sizes n=%d m=%d k=%d", n, m, k);
  KLLM_REQUIRE(dtype == DT_BF16 || dtype == DT_F32, "gemm_act: unknown dtype %d", dtype);
  const int chunk = dtype == DT_F32 ? 4 : 8;
  KLLM_REQUIRE(k % chunk == 0 && aligned16(x) && aligned16(w),
               "gemm_act: K=%d must be a multiple of %d and the operands 16-byte aligned", k, chunk);
  KLLM_REQUIRE((long)n * m < (1L << 31), "gemm_act: sizes overflow");
  if (int rc = gemm_ring(x, w, h, n, m, k, 1, RING_UNARY, dtype == DT_F32, dtype == DT_F32, act, act_params, stream)) return rc;
  KLLM_CHECK_LAUNCH("gemm_act");
  return 0;
}

// q = the rotated queries of x . w^T, keys and values into the pages: the product, the rotation and the append in one launch (RING_ROPE).
extern "C" int kllm_gemm_rope(const void* x, const KllmLinearOut* y, const void* w, int n, int m, int k, hipStream_t stream) {
  KLLM_REQUIRE(x && w && y && y->y && y->kind == KLLM_LINEAR_OUT_ROPE, "gemm_rope: null pointer, or another kind of output");
  KLLM_REQUIRE(n > 0 && m > 0 && k > 0, "gemm_rope: bad sizes n=%d m=%d k=%d", n, m, k);
  const int chunk = y->f32 ? 4 : 8, H = y->H, KV = y->KV, hd = y->hd;
  KLLM_REQUIRE(k % chunk == 0 && k < (1 << 23) && (long)m * k * (16 / chunk) < (1L << 32) && aligned16(x) && aligned16(w),
               "gemm_rope: K=%d must be a multiple of %d, the weights below 4 GiB and the operands 16-byte aligned", k, chunk);
  KLLM_REQUIRE(H > 0 && hd > 0 && hd % 8 == 0 && (!y->cache || KV > 0) && m == H * hd + (y->cache ? 2 * KV * hd : 0),
               "gemm_rope: m=%d does not fit %d and %d heads of %d (a multiple of 8)", m, H, KV, hd);
  KLLM_REQUIRE((y->cos_t == nullptr) == (y->sin_t == nullptr), "gemm_rope: cos and sin go together");
  KLLM_REQUIRE(aligned16(y->y) && aligned16(y->cache) && aligned16(y->cos_t) && aligned16(y->sin_t), "gemm_rope: unaligned pointer");
  KLLM_REQUIRE(!y->cache || (y->positions && y->span_of_token && y->block_table && y->max_pages > 0 && y->page_size > 0),
               "gemm_rope: the append needs positions, spans, a block table and pages");
  KLLM_REQUIRE((long)n * m < (1L << 31), "gemm_rope: sizes overflow");
  const RingRope rope = {y->cos_t, y->sin_t, y->cache, y->positions, y->span_of_token, y->block_table,
                         y->max_pages, y->page_size, H, y->cache ? KV : 0, hd / 2};
  if (int rc = gemm_ring(x, w, y->y, n, m / 2, k, 1, RING_ROPE, y->f32 != 0, y->f32 != 0, -1, nullptr, stream, rope)) return rc;
  KLLM_CHECK_LAUNCH("gemm_rope");
  return 0;
}
