// KV-cache decode split kernel on the matrix cores, for the 2 .. 8 query rows
// a KV head has with grouped-query heads (or a few new tokens).  Same work
// split, workspace and merge as decode_split_kernel (decode.hip): a workgroup
// reduces one split of the cache to partial (m, l, acc) rows.
//
// Why: on the vector units every row costs a key 16 multiplies and a
// cross-lane sum a lane, so from a few rows on the kernel is bound by them and
// not by HBM (4 rows, B64 Hkv8 D128 over 1025 f16 keys: 92 us for 268 MB, 2.9
// TB/s; over int8 codes 48 us for 66 MB).  Here a 32-key tile of D = 128 takes
// 8 MFMAs (16x16x32) for the scores and 24 for the values whatever the
// rows (up to 16, of which 2 .. 8 are used): about 500 cycles of one SIMD for
// 16 KB, which leaves the matrix cores 95% idle at HBM's rate.
//
// Measured in a kernel trace, vector kernel -> this one: that f16 case 92 -> 52
// us (5.2 TB/s), the int8 one 48 -> 23 us (2.8 TB/s, by the codes' conversion: 19
// vector instructions an MFMA).  K and V by non-temporal DMA were 3 - 5% slower.
// One row, and two over large caches (decode_mfma_applies), stay on the vector
// kernel, which reaches 6.5 TB/s there.
//
// Precision: q k products are exact in the MFMA and sum in fp32.  The
// probabilities are fp32 and stay so: each enters the value product as a sum
// of three f16 or bf16 numbers, one MFMA each over the same value fragment.
// The first two are truncated, so the three hold all 24 bits.  f16 parts are
// taken of P 2^14 (the factor cancels in acc / l): below P = 2^-15, where the
// last bits pass f16's smallest number, they are rounded at 2^-39 of the row's
// largest P.
//
// Every wave works alone on the tiles w, w + NWV, ... of the split through an LDS
// ring of its own (no barrier until the merge).  16-bit caches: K and V tiles
// come by DMA in the blocked layout of TileReader, three half-stages in flight
// (K of the next tile, V of this one and the next).  int8 caches: the codes
// come through registers, two tiles ahead, and are converted (exactly) to
// 16-bit tiles of the same layout; K's row scales multiply the scores, V's
// the probabilities.
#include <type_traits>

#include "decode_internal.h"
#include "rope_math.h"

namespace tsattn {
namespace {

constexpr int BN = 32;  // keys per tile

typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16x16x32, lane l = 16 g + c: A[c][8 g + j], B[8 g + j][c], j = 0..7;
// C[4 g + i][c], i = 0..3.
template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (std::is_same_v<T, bf16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Max over the four lanes c, c + 16, c + 32, c + 48 (v_permlane16_swap trades
// the odd 16-lane rows of one register for the even ones of the other).
__device__ __forceinline__ float quad_row_max(float x) {
  unsigned a = __builtin_bit_cast(unsigned, x), b = a;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return half_swap_max3(fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)));
}

// Waves per workgroup: 64 KiB of tiles, so two workgroups share a CU and one's
// prologue and merge run under the other's stream.
template <int D, bool Q8>
constexpr int dm_waves() {
  static_assert(!Q8 || D < 256, "int8 caches of 256 channels are the vector kernel's");
  return Q8 || D == 64 ? 4 : (D == 128 ? 2 : 1);
}

// x = hi + mid + lo, packed pairs of PT: hi and mid truncated, lo what is left.
template <typename PT>
struct Parts {
  static constexpr int N = 3;
  // The parts over values that may be infinite: where x != 0 none is 0 (0 * inf
  // would be NaN: f16's smallest number is 2^-38 of the row's largest P, bf16's
  // normal one nothing), and beside an infinite hi (int8 caches' scales are in x)
  // the others are finite.
  __device__ __forceinline__ static void fill(float a, float b, uint32_t (&out)[N]) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    constexpr uint16_t kTiny = std::is_same_v<PT, bf16> ? 0x0080 : 0x0001;
    const u16x2 least = {a != 0.f ? kTiny : uint16_t(0), b != 0.f ? kTiny : uint16_t(0)};
#pragma unroll
    for (int i = 0; i < N; ++i) {
      u16x2 x = __builtin_bit_cast(u16x2, out[i]);
      if (i > 0 && __builtin_isinf(a)) x[0] = 0;
      if (i > 0 && __builtin_isinf(b)) x[1] = 0;
      out[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(x, least));
    }
  }
  __device__ __forceinline__ static void split(float a, float b, uint32_t (&out)[N]) {
#pragma unroll
    for (int i = 0; i < N - 1; ++i) {
      if constexpr (std::is_same_v<PT, bf16>) {
        const uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
        out[i] = __builtin_amdgcn_perm(y, x, 0x07060302u);
        a -= __builtin_bit_cast(float, x & 0xFFFF0000u);
        b -= __builtin_bit_cast(float, y & 0xFFFF0000u);
      } else {
        out[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
        a -= static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(out[i])));
        b -= static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(out[i] >> 16)));
      }
    }
    out[N - 1] = pack2<PT>(a, b);
  }
};

// Eight int8 codes as eight values of T (exact).
template <typename T>
__device__ __forceinline__ u32x4 codes_to(u32x2 c) {
  u32x4 y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = c[i >> 1] >> (16 * (i & 1));
    y[i] = pack2<T>(static_cast<float>(static_cast<int8_t>(w & 0xFFu)),
                    static_cast<float>(static_cast<int8_t>((w >> 8) & 0xFFu)));
  }
  return y;
}

// MK: the problem has a mask (its element reads cost registers and code).
template <typename T, int D, bool Q8, bool MK>
__global__ __launch_bounds__((64 * dm_waves<D, Q8>()), (Q8 ? 2 : 1)) void decode_mfma_kernel(DecArgs a) {
  using KT = std::conditional_t<Q8, int8_t, T>;   // cache element type
  using PT = std::conditional_t<Q8, bf16, T>;     // value tiles and probability parts
  constexpr int NWV = dm_waves<D, Q8>();
  constexpr int NP = Parts<PT>::N;
  constexpr int SKS = D / 32;             // k-steps of S^T = K Q^T
  constexpr int PDT = D / 16;             // 16-row blocks of O^T
  constexpr int QG = D / 32;              // 4-chunk groups per row
  constexpr int TILE = BN * D * 2;        // bytes of a 16-bit K or V tile
  constexpr int BLK = TILE / 1024;        // DMA blocks per tile
  constexpr int WAVE_B = Q8 ? 2 * TILE + 256 : 4 * TILE;
  constexpr int ROWS = 8;                 // query rows at most
  constexpr int MERGE_B = NWV * ROWS * (D + 2) * 4;
  constexpr int LDS_B = NWV * WAVE_B > MERGE_B ? NWV * WAVE_B : MERGE_B;
  __shared__ __attribute__((aligned(1024))) char lds[LDS_B];

  const Problem &p = a.p;
  const int split = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int end = eff_end(p, b);
  const int k_begin = split * a.split_len;
  if (k_begin >= end) return;  // this split holds no keys for row b
  const int k_stop = min(k_begin + a.split_len, end);
  const int keys = __builtin_amdgcn_readfirstlane(k_stop - k_begin);
  const int n_tiles = (keys + BN - 1) / BN;
  const int mine = n_tiles > w ? (n_tiles - 1 - w) / NWV + 1 : 0;  // this wave's tiles
  // A key mask that is exactly the prefix [0, kv_len[b]) is already applied by k_stop.
  const bool masked = MK && !(p.kv_prefix && p.kv_prefix[b] && p.mask.s1 == 0 && p.mask.s2 == 0);

  // Lane (c, g): query row c = rr Sq + i (head hk rep + rr, position i), as the
  // B operand of S^T = K Q^T; rows past the last are zero and not stored.
  const int rr = c / p.Sq, qi = c - rr * p.Sq;
  const bool row_live = c < a.rows;
  u32x4 qf[SKS];
  {
    const T *qp = static_cast<const T *>(a.q.data) + b * a.q.s0 +
                  static_cast<int64_t>(row_live ? hk * p.rep + rr : 0) * a.q.s1 +
                  static_cast<int64_t>(row_live ? qi : 0) * a.q.s2 + 8 * g;
#pragma unroll
    for (int ks = 0; ks < SKS; ++ks) qf[ks] = ld16(qp + 32 * ks);
    if (p.rope.R > 0) {
      int64_t at[SKS];
      int p0[SKS];
#pragma unroll
      for (int ks = 0; ks < SKS; ++ks) {
        at[ks] = p.rope.qpos0 + (row_live ? qi : 0);
        p0[ks] = 16 * ks + 4 * g;
      }
      rotate_chunks<T, SKS>(qf, p.rope, at, p0, false);
    }
#pragma unroll
    for (int ks = 0; ks < SKS; ++ks) {
      if (!row_live) qf[ks] = u32x4{0, 0, 0, 0};
      asm volatile("" : "+v"(qf[ks]));  // loaded before the DMA stream starts
    }
  }

  // keys of the split this lane's row may see: [0, klim) of its own
  int klim = keys;
  if (p.causal) {
    const int64_t cl = static_cast<int64_t>(qi) + p.offset + 1 - k_begin;
    if (cl < klim) klim = cl < 0 ? 0 : static_cast<int>(cl);
  }
  const int edge = p.causal ? 0 : keys / BN;  // tiles from here on need the limit

  char *mylds = lds + w * WAVE_B;
  const uint32_t lds0 = lds_addr(lds) + w * WAVE_B;
  const uint32_t ks_b = static_cast<uint32_t>(a.k.s2) * sizeof(KT), vs_b = static_cast<uint32_t>(a.v.s2) * sizeof(KT);
  const KT *kbase = static_cast<const KT *>(a.k.data) + b * a.k.s0 + hk * a.k.s1 + static_cast<int64_t>(k_begin) * a.k.s2;
  const KT *vbase = static_cast<const KT *>(a.v.data) + b * a.v.s0 + hk * a.v.s1 + static_cast<int64_t>(k_begin) * a.v.s2;

  // Fragments of a tile in the blocked layout of TileReader (mfma_common.h):
  // K rows 16 kb + c, channels 32 ks + 8 g .. + 7; V^T channel 16 dt + c at the
  // keys 4 g .. + 3 and 16 + 4 g .. + 3, the order two score tiles hand over as
  // one B operand.
  const int koff_l = 4 * c * 16 + ((g ^ ((c >> 2) & 3)) << 4);
  int voff_l[2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
    voff_l[e] = ((4 * g + (c >> 2)) * 4 + ((2 * e + ((c & 3) >> 1)) ^ g)) * 16 + (c & 1) * 8;
  auto krows = [&](const char *tile, int kb, int ks) __attribute__((always_inline)) { return ld16(tile + (kb * QG + ks) * 1024 + koff_l); };
  auto vcols = [&](const char *tile, int dt) __attribute__((always_inline)) {
    const char *blk = tile + (dt >> 1) * 1024 + voff_l[dt & 1];
    const u32x2 x = ds_read_tr<PT>(reinterpret_cast<const PT *>(blk));
    const u32x2 y = ds_read_tr<PT>(reinterpret_cast<const PT *>(blk + QG * 1024));
    return u32x4{x[0], x[1], y[0], y[1]};
  };
  f32x4 oacc[PDT];
  // f16 parts are of P 2^14: the state's maximum is kept that much lower
  constexpr float kShift = std::is_same_v<PT, f16> ? 14.f : 0.f;
  float m, l;

  // Scores of the K tile at kt: element i is key 16 (i / 4) + 4 g + i % 4
  auto scores = [&](const char *kt, float (&x)[8]) __attribute__((always_inline)) {
    f32x4 s[2] = {f32x4{}, f32x4{}};
    u32x4 kf[2][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) kf[0][kb] = krows(kt, kb, 0);
#pragma unroll
    for (int ks = 0; ks < SKS; ++ks) {
      if (ks + 1 < SKS)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) kf[(ks + 1) & 1][kb] = krows(kt, kb, ks + 1);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] = mfma16<T>(kf[ks & 1][kb], qf[ks], s[kb]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = s[i >> 2][i & 3];
  };
  // Scores x (log2 units) of tile j -> the probabilities' parts; the running
  // maximum is raised (and l, acc rescaled) as the reference's recurrence does.
  // vsc: the tile's value scales (int8 caches).  filled: with Parts::fill.
  u32x4 pb[NP];
  auto softmax = [&](float (&x)[8], int j, const float *vsc, auto filled) __attribute__((always_inline)) {
    const int kv0 = j * BN;
    if (j >= edge || masked) {
      const int lim = klim - kv0 - 4 * g;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int kc = 16 * (i >> 2) + (i & 3);
        bool ok = kc < lim;
        if (MK && masked && ok && row_live) {
          const int64_t mi = b * p.mask.s0 + static_cast<int64_t>(hk * p.rep + rr) * p.mask.s1 +
                             static_cast<int64_t>(qi) * p.mask.s2 +
                             static_cast<int64_t>(k_begin + kv0 + 4 * g + kc) * p.mask.s3;
          if (p.mask.kind == TSATTN_MASK_BOOL) ok = static_cast<const uint8_t *>(p.mask.data)[mi] != 0;
          else x[i] += load_additive<float>(p.mask.data, mi, p.mask.dtype) * kLog2e;
        }
        if (!ok) x[i] = -INFINITY;
      }
    }
    float mx = x[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, x[i]);
    mx = quad_row_max(mx);
    if (__ballot(mx > m) != 0ull) {
      const float mn = fmaxf(m, mx);
      const float corr = mn == -INFINITY ? 1.f : fast_exp2(m - mn);
      m = mn;
      l *= corr;
#pragma unroll
      for (int dt = 0; dt < PDT; ++dt) oacc[dt] *= corr;
    }
    const float base = m == -INFINITY ? 0.f : kShift - m;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      float p0 = fast_exp2(x[i] + base), p1 = fast_exp2(x[i + 1] + base);
      l += p0 + p1;
      if constexpr (Q8) {
        p0 *= vsc[i];
        p1 *= vsc[i + 1];
      }
      uint32_t part[NP];
      Parts<PT>::split(p0, p1, part);
      if constexpr (decltype(filled)::value) Parts<PT>::fill(p0, p1, part);
#pragma unroll
      for (int n = 0; n < NP; ++n) pb[n][i >> 1] = part[n];
    }
  };
  // O^T += V^T P^T, every value fragment read once for the NP parts
  auto values = [&](const char *vt) __attribute__((always_inline)) {
    u32x4 vf[3];
    vf[0] = vcols(vt, 0);
    vf[1] = vcols(vt, 1);
#pragma unroll
    for (int dt = 0; dt < PDT; ++dt) {
      if (dt + 2 < PDT) vf[(dt + 2) % 3] = vcols(vt, dt + 2);
#pragma unroll
      for (int n = 0; n < NP; ++n) oacc[dt] = mfma16<PT>(vf[dt % 3], pb[n], oacc[dt]);
    }
  };

  // The wave's walk over its tiles.
  auto walk = [&](auto filled) __attribute__((always_inline)) {
#pragma unroll
  for (int dt = 0; dt < PDT; ++dt) oacc[dt] = f32x4{};
  m = -INFINITY, l = 0.f;
  if constexpr (!Q8) {
    const u32x4 kdesc = make_desc(kbase, static_cast<uint32_t>(keys) * ks_b);
    const u32x4 vdesc = make_desc(vbase, static_cast<uint32_t>(keys) * vs_b);
    const uint32_t chunk = (lane & 3) ^ ((lane >> 4) & 3);
    const uint32_t koff = (lane >> 2) * ks_b + chunk * 16, voff = (lane >> 2) * vs_b + chunk * 16;
    // local tile t (tile w + NWV t of the split) into stage t & 1; tiles past
    // the last read past the buffer range (zeros, no memory access)
    auto issue = [&](u32x4 desc, uint32_t off, uint32_t stride, int t, uint32_t half) __attribute__((always_inline)) {
      const uint32_t st = lds0 + static_cast<uint32_t>(t & 1) * 2 * TILE + half;
      const uint32_t row = t < mine ? static_cast<uint32_t>((w + NWV * t) * BN) * stride : 0x80000000u;
#pragma unroll
      for (int n = 0; n < BLK; ++n)
        dma16(desc, st + n * 1024, off, row + static_cast<uint32_t>(16 * (n / QG)) * stride + (n % QG) * 64);
    };
    issue(kdesc, koff, ks_b, 0, 0);
    issue(vdesc, voff, vs_b, 0, TILE);
    issue(kdesc, koff, ks_b, 1, 0);
    for (int t = 0; t < mine; ++t) {
      const char *kt = mylds + (t & 1) * 2 * TILE, *vt = kt + TILE;
      wait_vm_n<2 * BLK>();  // K of tile t has landed; V of t and K of t + 1 in flight
      __builtin_amdgcn_sched_barrier(0);
      float x[8];
      scores(kt, x);
      __builtin_amdgcn_sched_barrier(0);
      issue(vdesc, voff, vs_b, t + 1, TILE);  // (that stage's V was read for tile t - 1)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= a.sl;
      softmax(x, w + NWV * t, nullptr, filled);
      __builtin_amdgcn_sched_barrier(0);
      wait_vm_n<2 * BLK>();  // V of tile t; K and V of t + 1 in flight
      __builtin_amdgcn_sched_barrier(0);
      values(vt);
      wait_lgkm0();  // both tiles read
      __builtin_amdgcn_sched_barrier(0);
      issue(kdesc, koff, ks_b, t + 2, 0);
    }
    wait_vm_n<0>();
  } else {
    // codes of a tile: RPI rows per load, 8 codes a lane; lanes 0 .. 31 also
    // take the K scale of key `lane`, 32 .. 63 the V scales
    constexpr int LPR = D / 8, RPI = 64 / LPR, NL = BN / RPI;
    constexpr int RL = RPI < 4 ? RPI : 4;  // rows side by side in a lane group (bank spread)
    const int rest = lane / (4 * RL);
    const int lrow = ((lane >> 2) % RL) + RL * (rest / QG), lchunk = 4 * (rest % QG) + (lane & 3);
    const rsrc_t kr = make_rsrc(kbase, static_cast<uint32_t>(keys) * ks_b);
    const rsrc_t vr = make_rsrc(vbase, static_cast<uint32_t>(keys) * vs_b);
    const View &sv = lane < 32 ? a.ks : a.vs;
    const float *sp = static_cast<const float *>(sv.data) + b * sv.s0 + hk * sv.s1;
    float *scl = reinterpret_cast<float *>(mylds + 2 * TILE);  // [32 K scales | 32 V scales]
    struct Codes {
      u32x2 k[NL], v[NL];
      float sc;
    };
    auto load = [&](int t, Codes &x) __attribute__((always_inline)) {
      const int key0 = (w + NWV * t) * BN;
      const bool real = t < mine;
#pragma unroll
      for (int u = 0; u < NL; ++u) {
        const int key = key0 + u * RPI + lrow;
        const uint32_t dead = real ? 0u : 0x80000000u;
        x.k[u] = __builtin_amdgcn_raw_buffer_load_b64(kr, static_cast<int>((static_cast<uint32_t>(key) * ks_b + lchunk * 8) | dead), 0, 2);
        x.v[u] = __builtin_amdgcn_raw_buffer_load_b64(vr, static_cast<int>((static_cast<uint32_t>(key) * vs_b + lchunk * 8) | dead), 0, 2);
      }
      const int key = min(key0 + (lane & 31), keys - 1);  // (past the split: its last key, masked)
      x.sc = sp[static_cast<int64_t>(k_begin + key) * sv.s2];
    };
    auto compute = [&](int t, Codes &cd) __attribute__((always_inline)) {
      char *kt = mylds, *vt = mylds + TILE;
#pragma unroll
      for (int u = 0; u < NL; ++u) {
        const int r = u * RPI + lrow;
        const int at = ((r >> 4) * QG + (lchunk >> 2)) * 1024 + (4 * (r & 15) + ((lchunk & 3) ^ ((r >> 2) & 3))) * 16;
        *reinterpret_cast<u32x4 *>(kt + at) = codes_to<T>(cd.k[u]);
        *reinterpret_cast<u32x4 *>(vt + at) = codes_to<PT>(cd.v[u]);
      }
      scl[lane] = cd.sc;
      load(t + 2, cd);  // its registers are free now
      wait_lgkm0();    // (own wave's writes)
      __builtin_amdgcn_sched_barrier(0);
      float x[8], vsc[8];
      scores(kt, x);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const f32x4 k4 = *reinterpret_cast<const f32x4 *>(scl + 16 * e + 4 * g);
        const f32x4 v4 = *reinterpret_cast<const f32x4 *>(scl + 32 + 16 * e + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[4 * e + i] *= k4[i] * a.sl;
          vsc[4 * e + i] = v4[i];
        }
      }
      softmax(x, w + NWV * t, vsc, filled);
      values(vt);
      wait_lgkm0();  // the tile read before the next one overwrites it
      __builtin_amdgcn_sched_barrier(0);
    };
    Codes x0, x1;
    if (mine > 0) {
      load(0, x0);
      load(1, x1);
      for (int t = 0; t < mine; t += 2) {
        compute(t, x0);
        if (t + 1 < mine) compute(t + 1, x1);
      }
    }
  }
  };
  walk(std::false_type{});
  // sums that are not finite: again with filled parts (rare; its own code, so
  // that the first walk keeps its registers)
  float bad = 0.f;
#pragma unroll
  for (int dt = 0; dt < PDT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) bad = fmaf(oacc[dt][i], 0.f, bad);
  if (__ballot(bad != bad) != 0ull) walk(std::true_type{});

  // Merge the waves: [wave][row][D | m | l] in LDS, then every thread sums its
  // share of the outputs over the waves.
  float lt = l + __shfl_xor(l, 16, 64);
  lt += __shfl_xor(lt, 32, 64);
  const float ms = m == -INFINITY ? m : m - kShift;
  __syncthreads();  // every wave's tiles read
  float *part = reinterpret_cast<float *>(lds);
  if (row_live) {
    float *to = part + (w * ROWS + c) * (D + 2);
#pragma unroll
    for (int dt = 0; dt < PDT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) to[16 * dt + 4 * g + i] = oacc[dt][i];
    if (g == 0) {
      to[D] = ms;
      to[D + 1] = lt;
    }
  }
  __syncthreads();
  float *out = a.ws + (static_cast<int64_t>(b * p.Hkv + hk) * a.max_splits + split) * a.rows *
                          static_cast<int64_t>(D + 2);
  for (int idx = tid; idx < a.rows * (D + 2); idx += 64 * NWV) {
    const int r = idx / (D + 2), d = idx - r * (D + 2);
    const float *from = part + r * (D + 2);
    float M = -INFINITY;
#pragma unroll
    for (int v = 0; v < NWV; ++v) M = fmaxf(M, from[v * ROWS * (D + 2) + D]);
    const float base = M == -INFINITY ? 0.f : M;
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < NWV; ++v) {
      const float *f = from + v * ROWS * (D + 2);
      sum = fmaf(f[d], fast_exp2(f[D] - base), sum);
    }
    out[idx] = d == D ? M : sum;
  }
}

template <typename T, bool Q8>
void launch_t(const DecArgs &a, hipStream_t st) {
  const dim3 g(a.max_splits, a.p.Hkv, a.p.B);
  Probe pr_(Q8 ? "decode_mfma_int8" : "decode_mfma", st);
  auto run = [&](auto d, auto mk) {
    constexpr int D = decltype(d)::value;
    decode_mfma_kernel<T, D, Q8, decltype(mk)::value><<<g, dim3(64 * dm_waves<D, Q8>()), 0, st>>>(a);
  };
  auto dims = [&](auto mk) {
    if (a.p.Dqk == 64) run(std::integral_constant<int, 64>{}, mk);
    else if (a.p.Dqk == 128) run(std::integral_constant<int, 128>{}, mk);
    else if constexpr (!Q8) run(std::integral_constant<int, 256>{}, mk);
  };
  if (a.p.mask.kind == TSATTN_MASK_NONE) dims(std::false_type{});
  else dims(std::true_type{});
}

}  // namespace

bool decode_mfma_applies(const DecArgs &a, int dtype, bool q8) {
  if (dtype != TSATTN_F16 && dtype != TSATTN_BF16) return false;
  if (a.rows < 2 || a.rows > 8 || !(a.sl > 0.f) || !isfinite(a.sl)) return false;
  if (q8 && a.p.Dqk == 256) return false;  // (its codes, accumulators and parts exceed the registers)
  if (a.rows == 2) {
    // Two rows are few enough for the vector kernel to reach HBM's rate, and
    // then it is the faster one (16-bit, 64 sequences of 8 KV heads, 4000 keys: D64
    // 85 us, here 93; D128 173 and 186): it takes what the last-level cache does
    // not hold, 256 MiB (int8 at D128: half of that; 2000 keys 66 and 76 us), all of
    // D256 (4 sequences, 1000 keys: 13.2 and 14.6), and at D128 many heads of few
    // keys, which its shorter splits spread better (16 sequences, 1000 keys: 17.6
    // and 19.3).  The rest is faster here (D64, 16 x 8 heads, 4000 keys: 42 and 27;
    // int8 43 and 25; D128, 8 heads, 16000 keys: 31 and 21).
    const Problem &p = a.p;
    const int64_t heads = static_cast<int64_t>(p.B) * p.Hkv, mib = heads * p.Sk * p.Dqk * 2 * (q8 ? 1 : 2) >> 20;
    if (p.Dqk == 256 || mib >= (q8 && p.Dqk == 128 ? 128 : 256)) return false;
    if (p.Dqk == 128 && !q8 && heads >= 128 && p.Sk < 4000) return false;
  }
  // a split's rows are addressed with 32-bit offsets from its first key
  const int64_t es = q8 ? 1 : 2, most = static_cast<int64_t>(a.split_len) + 64;
  return a.k.s2 > 0 && a.v.s2 > 0 && most * a.k.s2 * es < (int64_t(1) << 31) &&
         most * a.v.s2 * es < (int64_t(1) << 31);
}

void launch_decode_mfma(const DecArgs &a, int dtype, bool q8, hipStream_t st) {
  if (dtype == TSATTN_BF16) {
    if (q8) launch_t<bf16, true>(a, st);
    else launch_t<bf16, false>(a, st);
  } else {
    if (q8) launch_t<f16, true>(a, st);
    else launch_t<f16, false>(a, st);
  }
}

}  // namespace tsattn
