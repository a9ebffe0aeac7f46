// What the two decode split kernels (decode.hip, decode_mfma.hip) share.
#pragma once

#include "mfma_common.h"

namespace tsattn {

struct DecArgs {
  Problem p;
  View q, k, v, o;
  View ks, vs;  // int8 caches: fp32 row scales [B, Hkv, capacity, 1]
  float *ws;
  int split_len, max_splits, rows;  // rows = rep * Sq query rows per KV head
  float sl;                         // scale * log2(e)
  bool mfma;                        // the matrix-core split kernel
};

// Keys any row may attend to: [0, eff_end).
__device__ __forceinline__ int eff_end(const Problem &p, int b) {
  int e = kv_end_for(p, b);
  if (p.causal) {
    const int64_t lim = static_cast<int64_t>(p.Sq) - 1 + p.offset + 1;
    if (lim < e) e = static_cast<int>(lim < 0 ? 0 : lim);
  }
  return e;
}

// Whether the matrix-core split kernel takes the problem (16-bit queries over
// a 16-bit or int8 cache, checked by decode_supported before), and its launch.
bool decode_mfma_applies(const DecArgs &a, int dtype, bool q8);
void launch_decode_mfma(const DecArgs &a, int dtype, bool q8, hipStream_t st);

}  // namespace tsattn
