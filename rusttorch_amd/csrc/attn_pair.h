// Prefill attention for head_dim 64 over f16 pairs; see attn_pair.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rtg {

// Power-of-two scales (gemm_pair.h: values times their scale are at most 2^15)
// per column; v's are also the output's. The products of a head's q and k
// scales are the same in all of its columns: qk[h], between 2^-100 and 2^110.
struct AttnScales {
  const float* q;   // [d]: c_attn's own
  const float* k;   // [d]
  const float* qk;  // [H]
  const float* v;   // [d]: c_attn's own
};
// k and qk from the scales col[2 d] of c_attn's q and k columns; *bad is set
// nonzero where a qk would be below 2^-100.
void launch_head_scale(hipStream_t s, const float* col, int H, float* k, float* qk, int* bad);

// S sequences of T new tokens at offset past: qkv rows [S * T][3 d] (q columns
// read), the cache of positions [0, past + T); out: pair matrix [S * T][d]
// scaled by sc.v.
void launch_attn_pair(hipStream_t s, const float* qkv, int S, int T, int past, const float* kc, const float* vc,
                      int n_head, int n_pos, int d, const AttnScales& sc, uint16_t* out);

}  // namespace rtg
