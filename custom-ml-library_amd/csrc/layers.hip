// The layers around the attention path, one kernel a pass: layer / RMS norm
// with its VJP (src/tensorsmith/nn/primitives.py:67-136) and the SwiGLU
// activation silu(gate) * up with its VJP (primitives.py:52-64 and
// src/tensorsmith/nn/transformer.py:190-205).  The reference writes each as a chain of array
// operations; run as such every link reads and writes the whole tensor.  All
// of them are bound by HBM (or, on a few rows, by the launch): each operand is
// read once and each result written once, 8 elements a lane and step.
//
// Half inputs compute in fp32 as the reference does; every value that the
// chain rounds to the tensor dtype (silu's result, the product's VJP) is
// rounded here too.
//
// A decoder block's training step (fp16 autocast, 8192 rows of 512, hidden
// 2048): 1534 us with the chains (8 launches a norm and 11 its VJP, 5 and 7 the
// activation), 1157 us with these (norm 10 us, its VJP 13 and the reduction 12);
// a 6-layer model's cached step on 4 rows, which the launches bound, 2399 -> 1611 us
// (and with the linear layers in rows.hip 315 - 350).
#include <type_traits>

#include "tsattn_internal.h"

namespace tsattn {
namespace {

constexpr int NT = 256;
constexpr int NW = NT / 64;
constexpr int VE = 8;  // elements a lane takes per step

template <typename T>
__device__ __forceinline__ void load8(const T *p, float (&x)[VE]) {
  typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
  constexpr int N = VE * sizeof(T) / 16;  // 16-byte loads
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const V y = *reinterpret_cast<const V *>(p + i * (16 / sizeof(T)));
#pragma unroll
    for (int e = 0; e < static_cast<int>(16 / sizeof(T)); ++e)
      x[i * (16 / sizeof(T)) + e] = static_cast<float>(y[e]);
  }
}
template <typename T>
__device__ __forceinline__ void store8(T *p, const float (&x)[VE]) {
  typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
  constexpr int N = VE * sizeof(T) / 16;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    V y;
#pragma unroll
    for (int e = 0; e < static_cast<int>(16 / sizeof(T)); ++e)
      y[e] = static_cast<T>(x[i * (16 / sizeof(T)) + e]);
    *reinterpret_cast<V *>(p + i * (16 / sizeof(T))) = y;
  }
}

__device__ __forceinline__ float wave_add(float x) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m, 64);
  return x;
}

// ---------------------------------------------------------------------------
// Norms.  A row belongs to one wave (G = 1, dim <= 2048) or to the workgroup's
// four (G = 4, dim <= 8192); lane l of wave w in the group takes the 8-element
// pieces w 64 + l + 64 G t, t < P = 4, and keeps them in registers between the
// statistics and the result.  Rows are walked by a grid that fills the chip
// once (the VJP's weight gradient then has few partial rows).
// ---------------------------------------------------------------------------
constexpr int P = 4;

struct NormArgs {
  int64_t rows;
  int dim;
  const void *x, *w, *bias, *g;
  void *out;           // forward: result; VJP: dx
  float *mean, *rstd;  // saved statistics (forward: NULL skips them)
  float *dw, *db;      // VJP: partial rows [gridDim.x][dim]
  float eps;
};

// sum over the G waves that share a row (every thread of the workgroup calls it)
template <int G>
__device__ __forceinline__ float row_sum(float x, float *red) {
  x = wave_add(x);
  if constexpr (G == 1) return x;
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = x;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < G; ++i) s += red[i];
  return s;
}

template <typename T, typename W, int G, bool RMS>
__global__ __launch_bounds__(NT) void norm_kernel(NormArgs a) {
  __shared__ float red[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int first = (G == 1 ? 0 : w) * 64 + lane;
  const float inv_dim = 1.f / static_cast<float>(a.dim);
  const int pieces = a.dim / VE;
  const int64_t step = static_cast<int64_t>(gridDim.x) * (NW / G);
  // (uniform trip count: with G = 4 every wave is on the same row)
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * (NW / G) + (G == 1 ? w : 0); r < a.rows; r += step) {
    const T *x = static_cast<const T *>(a.x) + r * a.dim;
    float v[P][VE];
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      const int pc = first + 64 * G * t;
#pragma unroll
      for (int e = 0; e < VE; ++e) v[t][e] = 0.f;
      if (pc < pieces) load8(x + pc * VE, v[t]);
#pragma unroll
      for (int e = 0; e < VE; ++e) s += v[t][e];
    }
    float mean = 0.f;
    if constexpr (!RMS) {
      mean = row_sum<G>(s, red) * inv_dim;
#pragma unroll
      for (int t = 0; t < P; ++t)
#pragma unroll
        for (int e = 0; e < VE; ++e) v[t][e] -= mean;
    }
    float q = 0.f;
#pragma unroll
    for (int t = 0; t < P; ++t)
      if (first + 64 * G * t < pieces)
#pragma unroll
        for (int e = 0; e < VE; ++e) q = fmaf(v[t][e], v[t][e], q);
    const float rstd = 1.f / sqrtf(row_sum<G>(q, red) * inv_dim + a.eps);
    T *out = static_cast<T *>(a.out) + r * a.dim;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      const int pc = first + 64 * G * t;
      if (pc >= pieces) continue;
      float wt[VE], y[VE];
      load8(static_cast<const W *>(a.w) + pc * VE, wt);
#pragma unroll
      for (int e = 0; e < VE; ++e) y[e] = v[t][e] * rstd * wt[e];
      if (a.bias) {
        float bt[VE];
        load8(static_cast<const W *>(a.bias) + pc * VE, bt);
#pragma unroll
        for (int e = 0; e < VE; ++e) y[e] += bt[e];
      }
      store8(out + pc * VE, y);
    }
    if (a.rstd && lane == 0 && (G == 1 || w == 0)) {
      a.rstd[r] = rstd;
      if constexpr (!RMS) a.mean[r] = mean;
    }
  }
}

// dx = rstd (g w - n mean(g w n)) (layer norm: - rstd mean(g w)), n the
// normalised row; dw = sum over rows of g n, db = sum of g, as one partial row
// per workgroup (norm_reduce_kernel adds them up in order: deterministic).
template <typename T, typename W, int G, bool RMS>
__global__ __launch_bounds__(NT) void norm_vjp_kernel(NormArgs a) {
  __shared__ float red[NW];
  __shared__ float part[G == 1 ? NW * 64 * VE : 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int first = (G == 1 ? 0 : w) * 64 + lane;
  const float inv_dim = 1.f / static_cast<float>(a.dim);
  const int pieces = a.dim / VE;
  const int64_t step = static_cast<int64_t>(gridDim.x) * (NW / G);
  float wt[P][VE], dw[P][VE], db[P][VE];
#pragma unroll
  for (int t = 0; t < P; ++t) {
    const int pc = first + 64 * G * t;
#pragma unroll
    for (int e = 0; e < VE; ++e) wt[t][e] = dw[t][e] = db[t][e] = 0.f;
    if (pc < pieces) load8(static_cast<const W *>(a.w) + pc * VE, wt[t]);
  }
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * (NW / G) + (G == 1 ? w : 0); r < a.rows; r += step) {
    const T *x = static_cast<const T *>(a.x) + r * a.dim;
    const T *g = static_cast<const T *>(a.g) + r * a.dim;
    const float rstd = a.rstd[r], mean = RMS ? 0.f : a.mean[r];
    float n[P][VE], gw[P][VE];
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      const int pc = first + 64 * G * t;
      if (pc < pieces) {
        load8(x + pc * VE, n[t]);
        load8(g + pc * VE, gw[t]);
      } else {
#pragma unroll
        for (int e = 0; e < VE; ++e) n[t][e] = mean, gw[t][e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        n[t][e] = (n[t][e] - mean) * rstd;
        dw[t][e] = fmaf(gw[t][e], n[t][e], dw[t][e]);
        if constexpr (!RMS) db[t][e] += gw[t][e];
        gw[t][e] *= wt[t][e];
        s1 = fmaf(gw[t][e], n[t][e], s1);
        if constexpr (!RMS) s2 += gw[t][e];
      }
    }
    s1 = row_sum<G>(s1, red) * inv_dim;
    if constexpr (!RMS) s2 = row_sum<G>(s2, red) * inv_dim;
    T *dx = static_cast<T *>(a.out) + r * a.dim;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      const int pc = first + 64 * G * t;
      if (pc >= pieces) continue;
      float y[VE];
#pragma unroll
      for (int e = 0; e < VE; ++e) y[e] = rstd * (gw[t][e] - n[t][e] * s1 - s2);
      store8(dx + pc * VE, y);
    }
  }
  float *dwp = a.dw + static_cast<int64_t>(blockIdx.x) * a.dim;
  float *dbp = a.db ? a.db + static_cast<int64_t>(blockIdx.x) * a.dim : nullptr;
  if constexpr (G != 1) {
#pragma unroll
    for (int t = 0; t < P; ++t) {
      const int pc = first + 64 * G * t;
      if (pc >= pieces) continue;
      store8(dwp + pc * VE, dw[t]);
      if (!RMS && dbp) store8(dbp + pc * VE, db[t]);
    }
  } else {
    // the four waves' sums of the same columns, in wave order
    auto flush = [&](const float (&acc)[P][VE], float *to) {
#pragma unroll
      for (int t = 0; t < P; ++t) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < VE; ++e) part[(w * VE + e) * 64 + lane] = acc[t][e];
        __syncthreads();
        // 512 columns of this step, two a thread
#pragma unroll
        for (int c = threadIdx.x; c < 64 * VE; c += NT) {
          const int col = 64 * VE * t + c;
          if (col >= a.dim) continue;
          float s = 0.f;
#pragma unroll
          for (int v = 0; v < NW; ++v) s += part[(v * VE + (c & (VE - 1))) * 64 + (c >> 3)];
          to[col] = s;
        }
      }
    };
    flush(dw, dwp);
    if (!RMS && dbp) flush(db, dbp);
  }
}

// out[col] = sum over the n partial rows, 64 columns and 16 slices of the rows
// per workgroup.
template <typename W>
__global__ __launch_bounds__(1024) void norm_reduce_kernel(const float *part, int n, int dim, W *out) {
  __shared__ float red[16][64];
  const int c = threadIdx.x & 63, sl = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
  float s = 0.f;
  if (col < dim)
    for (int r = sl; r < n; r += 16) s += part[static_cast<int64_t>(r) * dim + col];
  red[sl][c] = s;
  __syncthreads();
  if (sl == 0 && col < dim) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[i][c];
    out[col] = static_cast<W>(t);
  }
}

// ---------------------------------------------------------------------------
// SwiGLU activation: y = T(x sigmoid(x)), out = T(y u); VJP dup = T(g y),
// dgate = T(T(g u) (s + x s (1 - s))).
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ float round_to(float x) {
  return static_cast<float>(static_cast<T>(x));
}

template <typename T, bool VJP>
__global__ __launch_bounds__(NT) void silu_mul_kernel(const T *gate, const T *up, const T *g, T *out,
                                                      T *dup, int64_t pieces) {
  const int64_t step = static_cast<int64_t>(gridDim.x) * NT;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x; i < pieces; i += step) {
    float x[VE], u[VE], d[VE], o[VE];
    load8(gate + i * VE, x);
    load8(up + i * VE, u);
    if constexpr (VJP) load8(g + i * VE, d);
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      const float s = 1.f / (1.f + expf(-x[e]));
      const float y = round_to<T>(x[e] * s);
      if constexpr (VJP) {
        const float dy = round_to<T>(d[e] * u[e]);
        d[e] *= y;
        o[e] = dy * (s + x[e] * s * (1.f - s));
      } else {
        o[e] = y * u[e];
      }
    }
    store8(out + i * VE, o);
    if constexpr (VJP) store8(dup + i * VE, d);
  }
}

// Workgroups of a pass over `groups` units: one each, and from `most` on a
// workgroup walks several (its weights stay in registers).  On 256 CUs the norms
// run up to eight a CU, their VJP four (a partial weight-gradient row each, which
// norm_reduce_kernel reads: 11 us at 1024 rows of 512) and the activation 16.
unsigned grid_for(int64_t groups, int64_t most) {
  return static_cast<unsigned>(groups < 1 ? 1 : (groups < most ? groups : most));
}

template <typename T, typename W, int G>
void norm_rows(const NormArgs &a, bool rms, bool vjp, unsigned grid, hipStream_t st) {
  if (!vjp) {
    if (rms) norm_kernel<T, W, G, true><<<dim3(grid), dim3(NT), 0, st>>>(a);
    else norm_kernel<T, W, G, false><<<dim3(grid), dim3(NT), 0, st>>>(a);
  } else {
    if (rms) norm_vjp_kernel<T, W, G, true><<<dim3(grid), dim3(NT), 0, st>>>(a);
    else norm_vjp_kernel<T, W, G, false><<<dim3(grid), dim3(NT), 0, st>>>(a);
  }
}

template <typename T, typename W>
void norm_types(const NormArgs &a, bool rms, bool vjp, unsigned grid, hipStream_t st) {
  if (a.dim <= 64 * VE * P) norm_rows<T, W, 1>(a, rms, vjp, grid, st);
  else norm_rows<T, W, 4>(a, rms, vjp, grid, st);
}

template <typename T>
hipError_t norm_dispatch(const NormArgs &a, int w_dtype, bool rms, bool vjp, unsigned grid, hipStream_t st) {
  if (w_dtype == TSATTN_F32) norm_types<T, float>(a, rms, vjp, grid, st);
  else if (w_dtype == TSATTN_F16) norm_types<T, f16>(a, rms, vjp, grid, st);
  else norm_types<T, bf16>(a, rms, vjp, grid, st);
  return hipGetLastError();
}

hipError_t norm_any(const NormArgs &a, int dtype, int w_dtype, bool rms, bool vjp, unsigned grid, hipStream_t st) {
  if (dtype == TSATTN_F32) return norm_dispatch<float>(a, w_dtype, rms, vjp, grid, st);
  if (dtype == TSATTN_F16) return norm_dispatch<f16>(a, w_dtype, rms, vjp, grid, st);
  return norm_dispatch<bf16>(a, w_dtype, rms, vjp, grid, st);
}

// Rows the VJP gives one workgroup at least: its partial weight-gradient row
// costs as much traffic as one row of x.
int vjp_groups(int64_t rows, int dim) {
  const int64_t per = dim <= 64 * VE * P ? 4 * NW : 4;
  return static_cast<int>(grid_for((rows + per - 1) / per, 1024));
}

}  // namespace

size_t norm_workspace_bytes(int64_t rows, int dim, bool rms) {
  return static_cast<size_t>(vjp_groups(rows, dim)) * dim * (rms ? 1 : 2) * sizeof(float);
}

hipError_t launch_norm_forward(int dtype, int w_dtype, int64_t rows, int dim, bool rms, const void *x,
                               const void *w, const void *bias, void *out, float *mean, float *rstd,
                               double eps, hipStream_t st) {
  NormArgs a{rows, dim, x, w, bias, nullptr, out, mean, rstd, nullptr, nullptr, static_cast<float>(eps)};
  Probe pr_("norm", st);
  const int64_t per = dim <= 64 * VE * P ? NW : 1;
  return norm_any(a, dtype, w_dtype, rms, false, grid_for((rows + per - 1) / per, 2048), st);
}

hipError_t launch_norm_backward(int dtype, int w_dtype, int64_t rows, int dim, bool rms, const void *x,
                                const void *w, const void *g, const float *mean, const float *rstd,
                                void *dx, void *dw, void *db, float *ws, hipStream_t st) {
  const int n = vjp_groups(rows, dim);
  NormArgs a{rows, dim, x, w, nullptr, g, dx, const_cast<float *>(mean), const_cast<float *>(rstd), ws,
             rms ? nullptr : ws + static_cast<int64_t>(n) * dim, 0.f};
  {
    Probe pr_("norm_vjp", st);
    hipError_t e = norm_any(a, dtype, w_dtype, rms, true, static_cast<unsigned>(n), st);
    if (e != hipSuccess) return e;
  }
  Probe pr_("norm_reduce", st);
  const dim3 grid((dim + 63) / 64), blk(1024);
  for (int k = 0; k < (db ? 2 : 1); ++k) {
    const float *part = k ? a.db : a.dw;
    void *to = k ? db : dw;
    if (w_dtype == TSATTN_F32) norm_reduce_kernel<float><<<grid, blk, 0, st>>>(part, n, dim, static_cast<float *>(to));
    else if (w_dtype == TSATTN_F16) norm_reduce_kernel<f16><<<grid, blk, 0, st>>>(part, n, dim, static_cast<f16 *>(to));
    else norm_reduce_kernel<bf16><<<grid, blk, 0, st>>>(part, n, dim, static_cast<bf16 *>(to));
  }
  return hipGetLastError();
}

hipError_t launch_silu_mul(int dtype, int64_t n, const void *gate, const void *up, const void *g,
                           void *out, void *dup, hipStream_t st) {
  const int64_t pieces = n / VE;
  const dim3 grid(grid_for((pieces + NT - 1) / NT, 4096)), blk(NT);
  Probe pr_(g ? "silu_mul_vjp" : "silu_mul", st);
  auto run = [&](auto tag) {
    using T = decltype(tag);
    const T *x = static_cast<const T *>(gate), *u = static_cast<const T *>(up), *d = static_cast<const T *>(g);
    if (g) silu_mul_kernel<T, true><<<grid, blk, 0, st>>>(x, u, d, static_cast<T *>(out), static_cast<T *>(dup), pieces);
    else silu_mul_kernel<T, false><<<grid, blk, 0, st>>>(x, u, nullptr, static_cast<T *>(out), nullptr, pieces);
  };
  if (dtype == TSATTN_F32) run(float{});
  else if (dtype == TSATTN_F16) run(f16{});
  else run(bf16{});
  return hipGetLastError();
}

}  // namespace tsattn
