// gemm_sb_api.hpp -- launch interface of the K-quant prefill GEMM (gemm_sb.hpp).
#pragma once

#include "wh_common.hpp"

namespace wh {

struct SbGemm {
  const uint8_t* w;        // stage records (kquant_repacked_bytes)
  const uint8_t* w2;       // ffn: the up matrix (w is the gate)
  const _Float16* frag;    // packed activations, row scales and (Q4_K) super-block sums
  const float* rs;
  const float* bs;
  float* y;                // output; with splits > 1 that many planes of it
  int n_tokens, n_rows, k, bm, splits;
  bool ffn;                // y = silu(w x) * (w2 x)
  bool lo;                 // false: bf16 activations, whose lo limbs are zero
  uint32_t* sk_flags;      // stream-K: flags, partial tiles, workgroups (0: a workgroup per tile)
  float* sk_part;
  int sk_g, sk_sub;
  uint32_t sk_wait;
};
int launch_gemm_sb_q4(const SbGemm& a, hipStream_t s);
int launch_gemm_sb_q6(const SbGemm& a, hipStream_t s);

}  // namespace wh
