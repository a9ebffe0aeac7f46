// Weight gradient of a linear layer, dW[m][n] = sum_t G[t][m] X[t][n] over many
// tokens (src/tensorsmith/nn/functional.py:63-90, the VJP's grad^T @ input), f16
// / bf16 in, fp32 sums, dW rounded to the dtype once.
//
// The output is small (a few tiles) and the contraction long: one workgroup per
// output tile leaves most of the chip idle (512 x 512 over 8192 tokens is 16
// tiles of 128), so the tokens split over `splits` workgroups a tile, whose fp32
// partial tiles a second kernel adds up in order (deterministic).  Bound by the
// matrix cores' operand reads: both operands are wanted along the token axis,
// so every fragment is two LDS transpose reads, and a 64 x 64 wave tile needs
// eight for four MFMAs, which is about what the LDS delivers in that time.
//
// Workgroup = 128 x 128 outputs, 4 waves x (64 x 64); stages of 32 tokens (G | X,
// 16 KiB) in a 4-stage ring, DMA three ahead, one fence-free barrier a stage; two
// workgroups a CU.  Consecutive workgroups (different XCDs) take different
// token ranges, so each XCD's L2 holds its own range of G and X only.
//
// Measured over 8192 tokens, against the library's product: 512 x 512 20 us (53),
// 2048 x 512 31 us (55), 768 x 768 24 us (49), 1024 x 1024 30 us (56); a decoder
// block's training step (512 wide, hidden 2048, 8192 rows) 1157 -> 1112 us, its kernels
// 1160 -> 890 us (the host bounds the rest).
#include "mfma_common.h"

namespace tsattn {
namespace {

constexpr int NT = 256;
constexpr int BT = 32;    // tokens per stage
constexpr int BM = 128;   // output tile edge
constexpr int NS = 4;     // ring stages
constexpr int TILE = BT * BM * 2;
constexpr int STAGE = 2 * TILE;

struct WgradArgs {
  int tokens, M, N, per;    // per: tokens a split takes (a multiple of BT)
  int splits;
  const void *g, *x;
  int64_t gs, xs;           // row strides (elements)
  float *part;              // [splits][M][N]
};

template <typename T>
__global__ __launch_bounds__(NT, 2) void wgrad_kernel(WgradArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nt_n = (a.N + BM - 1) / BM;
  const int split = blockIdx.x % a.splits, tile = blockIdx.x / a.splits;
  const int m0 = tile / nt_n * BM, n0 = tile % nt_n * BM;
  const int t0 = split * a.per, count = min(a.per, a.tokens - t0);  // (>= 1: the host sizes splits so)
  const int stages = (count + BT - 1) / BT;

  // the split's rows of each operand; tokens past the last read as zeros
  const uint32_t gs_b = static_cast<uint32_t>(a.gs) * 2, xs_b = static_cast<uint32_t>(a.xs) * 2;
  const u32x4 gdesc = make_desc(static_cast<const T *>(a.g) + static_cast<int64_t>(t0) * a.gs,
                                static_cast<uint32_t>(count - 1) * gs_b + static_cast<uint32_t>(a.M) * 2);
  const u32x4 xdesc = make_desc(static_cast<const T *>(a.x) + static_cast<int64_t>(t0) * a.xs,
                                static_cast<uint32_t>(count - 1) * xs_b + static_cast<uint32_t>(a.N) * 2);
  // Blocked layout (TileReader): block n = (16-token group n / 4, 64-byte column
  // group n % 4); wave w loads column group w of both token groups of both
  // operands.  Columns past the last read as zeros (offsets past the range).
  const uint32_t chunk = (lane & 3) ^ ((lane >> 4) & 3);
  const int col = 32 * w + 8 * static_cast<int>(chunk);  // the lane's first column in the tile
  const uint32_t goff = (static_cast<uint32_t>(lane >> 2) * gs_b + static_cast<uint32_t>(m0 + col) * 2) |
                        (m0 + col < a.M ? 0u : 0x80000000u);
  const uint32_t xoff = (static_cast<uint32_t>(lane >> 2) * xs_b + static_cast<uint32_t>(n0 + col) * 2) |
                        (n0 + col < a.N ? 0u : 0x80000000u);
  const uint32_t lds0 = lds_addr(lds);
  auto issue = [&](int s) {  // 4 loads a wave; past the last stage: zeros, no memory access
    const uint32_t st = lds0 + static_cast<uint32_t>(s % NS) * STAGE + w * 1024;
    const uint32_t far = s < stages ? 0u : 0x80000000u;
#pragma unroll
    for (int rg = 0; rg < 2; ++rg) {
      const uint32_t row = static_cast<uint32_t>(s < stages ? s * BT + 16 * rg : 0);
      dma16(gdesc, st + rg * 4096, goff | far, row * gs_b);
      dma16(xdesc, st + TILE + rg * 4096, xoff | far, row * xs_b);
    }
  };
  const TileReader<T, BM> rd(lane);
  const int wm = w >> 1, wn = w & 1;  // 64 x 64 quarter of the tile
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};

#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s);
  for (int s = 0; s < stages; ++s) {
    wait_vm_n<4 * (NS - 2)>();  // this wave's part of stage s has landed
    phase_barrier();            // ... and every wave's; stage s - 1 is read by all
    issue(s + NS - 1);          // into stage s - 1's slot
    const char *gt = lds + (s % NS) * STAGE, *xt = gt + TILE;
    u32x4 fa[2][2], fb[2][2];
    auto load = [&](int ks) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[ks][i] = rd.cols(gt, ks, 2 * wm + i);
        fb[ks][i] = rd.cols(xt, ks, 2 * wn + i);
      }
    };
    load(0);
    load(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32<T>(fa[ks][i], fb[ks][j], acc[i][j]);
    wait_lgkm0();
  }
  wait_vm_n<0>();
  // lane holds C[m = 8 (e / 4) + 4 h + e % 4][n = c] of each 32 x 32 block
  float *out = a.part + static_cast<int64_t>(split) * a.M * a.N;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + 64 * wn + 32 * j + c;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + 64 * wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
        if (m < a.M && n < a.N) out[static_cast<int64_t>(m) * a.N + n] = acc[i][j][e];
      }
    }
}

// dW = the splits' partial sums, four elements a thread.  Up to 8 splits: one
// thread adds them all.  More: the workgroup's four waves take every 4th split
// of the same 64 pieces, eight loads in flight each, and add up in order (512 x
// 512, 16 splits: 7 -> 4 us; at 4 splits the extra workgroups cost 2 us).
//
// O: T, or float for a parameter kept in fp32 -- the sum rounded to T all the
// same, as a T gradient widened afterwards would be, without that pass.
template <typename T, typename O, int G>
__global__ __launch_bounds__(NT) void wgrad_reduce_kernel(const float *part, int splits, int64_t n4, O *out) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int PER = NT / G;  // pieces per workgroup
  __shared__ f4 red[G][PER];
  const int lane = threadIdx.x % PER, grp = threadIdx.x / PER;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * PER + lane, ii = i < n4 ? i : n4 - 1;
  const f4 *p = reinterpret_cast<const f4 *>(part) + ii;
  f4 s = f4{};
  constexpr int U = 8;
  for (int k0 = grp; k0 < splits; k0 += G * U) {
    f4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = p[static_cast<int64_t>(min(k0 + G * u, splits - 1)) * n4];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + G * u < splits) s += v[u];
  }
  if constexpr (G > 1) {
    red[grp][lane] = s;
    __syncthreads();
    if (grp != 0) return;
#pragma unroll
    for (int k = 1; k < G; ++k) s += red[k][lane];
  }
  if (i >= n4) return;
  if constexpr (sizeof(O) == 4) {
    f4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = static_cast<float>(static_cast<T>(s[e]));
    *reinterpret_cast<f4 *>(out + 4 * i) = r;
  } else {
    *reinterpret_cast<u32x2 *>(out + 4 * i) = u32x2{pack2<T>(s[0], s[1]), pack2<T>(s[2], s[3])};
  }
}

// About one workgroup a CU (256): at two a CU the partial tiles' traffic doubles
// and costs more than the second workgroup hides (8192 tokens, 512 x 512: 20 us
// against 25).  A number that divides the eight XCDs keeps each token range in
// the L2s of the same XCDs; three, or five to seven, has every L2 read them all
// (16384 tokens: 1024 x 1408, 3 splits 120 us, 4 58, the library's product 114; 768
// x 1280, 5 splits 82, 8 41, the library 100).  Tiles past half of the CUs take 4 too
// (1536 x 1536, 65536 tokens: 2 splits 528 us, 4 479).
int wgrad_splits(int tokens, int M, int N) {
  const int64_t tiles = static_cast<int64_t>((M + BM - 1) / BM) * ((N + BM - 1) / BM);
  int64_t s = tiles >= 64 ? 4 : (tiles > 32 ? 8 : (256 + tiles - 1) / tiles);
  const int64_t most = (tokens + 4 * BT - 1) / (4 * BT);  // at least four stages a split
  if (s > most) s = most;
  if (s < 1) s = 1;
  const int per = static_cast<int>(((tokens + s - 1) / s + BT - 1) / BT * BT);
  return (tokens + per - 1) / per;
}

}  // namespace

size_t wgrad_workspace_bytes(int tokens, int M, int N) {
  return static_cast<size_t>(wgrad_splits(tokens, M, N)) * M * N * sizeof(float);
}

hipError_t launch_wgrad(int dtype, int out_dtype, int tokens, int M, int N, const void *g, int64_t gs, const void *x,
                        int64_t xs, void *dw, float *ws, hipStream_t st) {
  const int splits = wgrad_splits(tokens, M, N);
  const int per = ((tokens + splits - 1) / splits + BT - 1) / BT * BT;
  WgradArgs a{tokens, M, N, per, splits, g, x, gs, xs, ws};
  const int tiles = ((M + BM - 1) / BM) * ((N + BM - 1) / BM);
  const int64_t n4 = static_cast<int64_t>(M) * N / 4;
  const dim3 grid(tiles * splits), blk(NT);
  {
    Probe pr_("wgrad", st);
    if (dtype == TSATTN_BF16) wgrad_kernel<bf16><<<grid, blk, 0, st>>>(a);
    else wgrad_kernel<f16><<<grid, blk, 0, st>>>(a);
  }
  Probe pr_("wgrad_reduce", st);
  auto reduce = [&](auto tag, auto otag) {
    using T = decltype(tag);
    using O = decltype(otag);
    O *out = static_cast<O *>(dw);
    if (splits > 8)
      wgrad_reduce_kernel<T, O, 4><<<dim3(static_cast<unsigned>((n4 + 63) / 64)), blk, 0, st>>>(ws, splits, n4, out);
    else
      wgrad_reduce_kernel<T, O, 1>
          <<<dim3(static_cast<unsigned>((n4 + NT - 1) / NT)), blk, 0, st>>>(ws, splits, n4, out);
  };
  if (dtype == TSATTN_BF16) out_dtype == TSATTN_F32 ? reduce(bf16{}, 0.f) : reduce(bf16{}, bf16{});
  else out_dtype == TSATTN_F32 ? reduce(f16{}, 0.f) : reduce(f16{}, f16{});
  return hipGetLastError();
}

}  // namespace tsattn
