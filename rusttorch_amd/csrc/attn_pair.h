// Prefill attention for head_dim 64 over f16 pairs; see attn_pair.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rtg {

// Power-of-two scales (gemm_pair.h: values times their scale are at most 2^15):
// of q and k per head, of v per column; v's are also the output's.
struct AttnScales {
  const float* q;
  const float* k;
  const float* v;
};
// q[h], k[h] from the scales col[2 d] of c_attn's q and k columns, their product
// between 2^-100 and 2^110; *bad is set nonzero where it would be smaller.
void launch_head_scale(hipStream_t s, const float* col, int H, float* q, float* k, int* bad);

// S sequences of T new tokens at offset past: qkv rows [S * T][3 d] (q columns
// read), the cache of positions [0, past + T); out: pair matrix [S * T][d]
// scaled by sc.v.
void launch_attn_pair(hipStream_t s, const float* qkv, int S, int T, int past, const float* kc, const float* vc,
                      int n_head, int n_pos, int d, const AttnScales& sc, uint16_t* out);

}  // namespace rtg
