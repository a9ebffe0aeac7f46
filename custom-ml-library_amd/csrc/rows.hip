// Linear layers over few rows (the cached decode step: one row per stream):
// out[r][n] = sum_k x[r][k] W[n][k], W row-major as Linear.weight
// (src/tensorsmith/nn/functional.py:63-90), with what the decoder block does to the result folded
// in: the bias, the residual sum (transformer.py:226-243), or for a pair of
// weights the SwiGLU activation silu(gate) * up (transformer.py:190-205).  Every value the separate
// ops round to the dtype is rounded here too.
//
// Bound by the weights' stream (N K 2 bytes from HBM once; the rows stay in L2)
// and on small layers by the launch and one memory round trip.  One workgroup =
// 32 output channels x 32 rows; its NW waves take the 64-column chunks of K in
// turn, each through an LDS ring of its own filled by DMA three chunks ahead
// (whole 128-byte lines, eight rows an instruction), 8 KiB a chunk: W and x
// rows.  Chunk ch goes to accumulator ch % 8 and the eight sum in order, as in
// the fused projection kernel (qkv.hip), so the products do not depend on NW.
// NW = 4 keeps 128 KiB in flight on the CU a workgroup has to itself (layers
// with fewer tiles than the chip takes at two a CU), NW = 2 runs two a CU.
//
// Measured (f16, cold weights): K 512, N 512 .. 2048 4.2 us; 2048 x 2048 5.7;
// 4096 x 4096 10.6 (3.2 TB/s; 64 rows 12.8); 4096 x 16384 29.7 us (4.5 TB/s).  The library's product
// takes 12 us on the GPU at 4096 x 4096 and 64 rows and 18 us of host time a call,
// which bounds it on every smaller layer.  The 6-layer model's cached step on 4
// rows, with a block's step in one call: 1611 -> 315 - 350 us (51 launches, 238 us of GPU
// time); the attention layer's over int8 codes (B16 E2048, 4001 positions) 94 -> 41 us.
#include <type_traits>

#include "mfma_common.h"

namespace tsattn {
namespace {

constexpr int NACC = 8;   // chunk accumulators (summed in order)
constexpr int NSTG = 4;   // ring stages per wave

struct RowsArgs {
  int rows, K, n[3];        // outputs of the (up to three) weights, one after another in a row of out
  const void *x, *w[3], *bias[3], *res;
  void *out;
  int64_t xs, rs, os;       // element strides between rows of x, res and out
};

__device__ __forceinline__ const void *uniform_ptr(const void *p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const void *>((static_cast<uint64_t>(hi) << 32) | lo);
}

// DUAL: w[0] and w[1] are gate and up, half of the waves each.
template <typename T, int NW, bool DUAL>
__global__ __launch_bounds__(64 * NW) void rows_linear_kernel(RowsArgs a) {
  constexpr int MATS = DUAL ? 2 : 1;
  constexpr int WPM = NW / MATS;            // waves per matrix
  constexpr int APW = NACC / WPM;           // accumulators per wave
  constexpr int RING = NSTG * 8192;
  constexpr int PART = MATS * NACC * 16 * 64 * 4;
  __shared__ __attribute__((aligned(1024))) char smem[NW * RING > PART ? NW * RING : PART];
  auto part = reinterpret_cast<float (*)[NACC][16][64]>(smem);

  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mat = DUAL ? w / WPM : 0, wm = DUAL ? w % WPM : w;
  // the row blocks of a weight tile are consecutive and share an XCD's L2
  const int rblocks = (a.rows + 31) / 32;
  const int logical = xcd_remap(blockIdx.x, static_cast<int>(gridDim.x));
  const int rb = logical % rblocks;
  int tile = logical / rblocks, seg = 0, base = 0;  // 32-channel tile of weight `seg`
  if constexpr (!DUAL) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int t = (a.n[s] + 31) / 32;
      if (seg == s && tile >= t) {
        tile -= t;
        base += a.n[s];
        seg = s + 1;
      }
    }
  }
  const int n0 = 32 * tile, r0 = 32 * rb;
  const int nn = seg == 0 ? a.n[0] : (seg == 1 ? a.n[1] : a.n[2]);
  const int wsel = DUAL ? mat : seg;
  const void *wp = wsel == 0 ? a.w[0] : (wsel == 1 ? a.w[1] : a.w[2]);
  const T *W = static_cast<const T *>(uniform_ptr(static_cast<const T *>(wp) + static_cast<int64_t>(n0) * a.K));
  const int wrows = min(32, nn - n0);  // channels past the last read as zeros

  f32x16 acc[APW];
#pragma unroll
  for (int v = 0; v < APW; ++v) acc[v] = f32x16{};
  {
    const uint32_t sbase = lds_addr(smem) + w * RING;
    const int nch = (a.K + 63) / 64;
    const int mine = nch > wm ? (nch - 1 - wm) / WPM + 1 : 0;  // this wave's chunks
    const int lr = lane >> 3, gu = (lane & 7) ^ lr;  // row within 8, 16-byte unit of the chunk
    const u32x4 wdesc = make_desc(W, static_cast<uint32_t>(wrows) * a.K * 2);
    const int64_t xext = (static_cast<int64_t>(a.rows) - 1) * a.xs + a.K;
    const u32x4 xdesc = make_desc(uniform_ptr(a.x), static_cast<uint32_t>(xext * 2));
    uint32_t wv[4], xv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 8 * i + lr;
      wv[i] = (static_cast<uint32_t>(row) * a.K + 8 * gu) * 2;
      const int xr = r0 + row;
      xv[i] = (static_cast<uint32_t>(static_cast<int64_t>(min(xr, a.rows - 1)) * a.xs + 8 * gu) * 2) |
              (xr < a.rows ? 0u : 0x80000000u);  // rows past the last read as zeros
    }
    // chunk k of this wave (past its last: zeros, no memory access) into the stage at st
    auto issue = [&](int k, uint32_t st) {
      const int ch = wm + WPM * k;
      const bool real = k < mine;
      const uint32_t col = static_cast<uint32_t>(ch) * 64 + 8 * gu;
      const uint32_t far = (real && col < static_cast<uint32_t>(a.K)) ? 0u : 0x80000000u;
      const uint32_t soff = real ? static_cast<uint32_t>(ch) * 128 : 0u;
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(wdesc, st + i * 1024, wv[i] | far, soff);
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(xdesc, st + 4096 + i * 1024, xv[i] | far, soff);
    };
    const uint32_t fo = static_cast<uint32_t>(c) * 128;
    const uint32_t last = sbase + (NSTG - 1) * 8192;
    uint32_t ist = sbase;
    int rd = 0;
    auto step = [&](int k, f32x16 &ac) {
      issue(k + NSTG - 1, ist);
      ist = ist == last ? sbase : ist + 8192;
      wait_vm_n<8 * (NSTG - 1)>();  // chunk k has landed; the next chunks' loads stay in flight
      __builtin_amdgcn_sched_barrier(0);
      const char *stg = smem + w * RING + rd;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint32_t u = static_cast<uint32_t>((2 * s + h) ^ (c & 7)) * 16;
        const u32x4 wf = *reinterpret_cast<const u32x4 *>(stg + fo + u);
        const u32x4 xf = *reinterpret_cast<const u32x4 *>(stg + 4096 + fo + u);
        ac = mfma32<T>(wf, xf, ac);
      }
      wait_lgkm0();  // reads of this stage done before chunk k + NSTG overwrites it
      __builtin_amdgcn_sched_barrier(0);
      rd = rd == (NSTG - 1) * 8192 ? 0 : rd + 8192;
    };
#pragma unroll
    for (int k = 0; k < NSTG - 1; ++k) {
      issue(k, ist);
      ist = ist == last ? sbase : ist + 8192;
    }
    for (int k = 0; k < mine; k += APW) {
#pragma unroll
      for (int v = 0; v < APW; ++v)
        if (k + v < mine) step(k + v, acc[v]);
    }
    wait_vm_n<0>();
    __syncthreads();  // every ring read before the partial tiles reuse the LDS
  }
#pragma unroll
  for (int v = 0; v < APW; ++v)
#pragma unroll
    for (int e = 0; e < 16; ++e) part[mat][wm + WPM * v][e][lane] = acc[v][e];
  __syncthreads();

  // channel group g of 8: lane (c, h) holds channels n0 + 8 g + 4 h .. + 3 of row r0 + c
  const int r = r0 + c;
  for (int g = w; g < 4; g += NW) {
    const int n = n0 + 8 * g + 4 * h;
    if (r >= a.rows || n >= nn) continue;
    const T *bias = static_cast<const T *>(seg == 0 ? a.bias[0] : (seg == 1 ? a.bias[1] : a.bias[2]));
    T y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float s[MATS];
#pragma unroll
      for (int t = 0; t < MATS; ++t) {
        s[t] = 0.f;
#pragma unroll
        for (int v = 0; v < NACC; ++v) s[t] += part[t][v][4 * g + e][lane];
      }
      // the product in the dtype, then each op on it in the dtype
      y[e] = static_cast<T>(s[0]);
      if constexpr (DUAL) {
        const float x = static_cast<float>(y[e]);
        const T act = static_cast<T>(x * (1.f / (1.f + expf(-x))));
        y[e] = static_cast<T>(static_cast<float>(act) * static_cast<float>(static_cast<T>(s[1])));
      } else if (bias) {
        y[e] = static_cast<T>(static_cast<float>(y[e]) + static_cast<float>(bias[n + e]));
      }
    }
    const int64_t at = base + n;
    if (a.res) {
      const T *rp = static_cast<const T *>(a.res) + r * a.rs + at;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = static_cast<T>(static_cast<float>(rp[e]) + static_cast<float>(y[e]));
    }
    auto bits = [&](int e) { return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, y[e])); };
    *reinterpret_cast<u32x2 *>(static_cast<T *>(a.out) + r * a.os + at) =
        u32x2{bits(0) | (bits(1) << 16), bits(2) | (bits(3) << 16)};
  }
}

template <typename T>
void launch_t(const RowsArgs &a, bool dual, int tiles, hipStream_t st) {
  const int grid = tiles * ((a.rows + 31) / 32);
  if (dual) rows_linear_kernel<T, 4, true><<<dim3(grid), dim3(256), 0, st>>>(a);
  else if (grid < 512) rows_linear_kernel<T, 4, false><<<dim3(grid), dim3(256), 0, st>>>(a);
  else rows_linear_kernel<T, 2, false><<<dim3(grid), dim3(128), 0, st>>>(a);
}

}  // namespace

hipError_t launch_rows_linear(int dtype, int rows, int K, const int n[3], const void *x, int64_t xs,
                              const void *const w[3], const void *const bias[3], const void *res, int64_t rs,
                              void *out, int64_t os, hipStream_t st) {
  RowsArgs a{rows, K, {n[0], n[1], n[2]}, x, {w[0], w[1], w[2]}, {bias[0], bias[1], bias[2]}, res, out, xs, rs, os};
  const int tiles = (n[0] + 31) / 32 + (n[1] + 31) / 32 + (n[2] + 31) / 32;
  Probe pr_("rows_linear", st);
  if (dtype == TSATTN_BF16) launch_t<bf16>(a, false, tiles, st);
  else launch_t<f16>(a, false, tiles, st);
  return hipGetLastError();
}

hipError_t launch_rows_swiglu(int dtype, int rows, int K, int N, const void *x, int64_t xs, const void *gate,
                              const void *up, void *out, int64_t os, hipStream_t st) {
  RowsArgs a{rows, K, {N, 0, 0}, x, {gate, up, nullptr}, {nullptr, nullptr, nullptr}, nullptr, out, xs, 0, os};
  Probe pr_("rows_swiglu", st);
  if (dtype == TSATTN_BF16) launch_t<bf16>(a, true, (N + 31) / 32, st);
  else launch_t<f16>(a, true, (N + 31) / 32, st);
  return hipGetLastError();
}

}  // namespace tsattn
