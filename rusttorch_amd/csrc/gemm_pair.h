// Prefill GEMM on f16 MFMA over f16 pairs (f16_pair.h); see gemm_pair.hip for
// the arithmetic and the tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace rtg {

// One weight matrix W^T [N][K] (K % 64 == 0) as f16 operands. Column k of the
// input it multiplies is held scaled by in_scale[k], so W holds
// W[n][k] / in_scale[k], scaled to row n's own power of two; a product of the
// two is y[n] / out_scale[n].
struct PairWeights {
  uint16_t* w = nullptr;       // planes 2: rows of K / 32 groups [32 hi][32 lo]; planes 1: rows of K f16
  int planes = 2;              // 2: f32 weights, 1: bf16 weights (8 significant bits fit one f16)
  int N = 0, K = 0;
  float* out_scale = nullptr;  // [N], powers of two
};

// Bytes of PairWeights::w.
size_t pair_weight_bytes(int N, int K, int wtype);

// Power-of-two input scales. pair_ln_scale: of LN(x) with gain g and bias b,
// |LN(x)_k| <= sqrt(d) |g_k| + |b_k| for every x. pair_row_scale: of the
// outputs W[n] . LN(x) + bias[n] of a GEMM over that LayerNorm's output (and
// of anything no larger: averages over rows, gelu), by Cauchy-Schwarz at most
// sqrt(K) |W[n] * g|_2 + |W[n] . b + bias[n]|. Each value times its scale is
// at most 2^15 in magnitude, half of f16's range. *bad is set nonzero where a
// bound is 2^95 or more, or not a number.
void launch_pair_ln_scale(hipStream_t s, const float* g, const float* b, int d, float* scale, int* bad);
void launch_pair_row_scale(hipStream_t s, const void* W, int wtype, int N, int K, const float* g, const float* b,
                           const float* bias, float* scale, int* bad);
// Fills pw->w and pw->out_scale (both allocated) from row-major W^T.
void launch_pair_weights(hipStream_t s, const void* W, int wtype, const float* in_scale, const PairWeights& pw,
                         int* bad);

struct PairGemmArgs {
  const uint16_t* A = nullptr;  // pair matrix [M][K] (pair_index), input columns scaled
  long lda = 0;                 // row stride in f16 elements (2 K for consecutive rows)
  int M = 0;
  const float* bias = nullptr;  // [N] or null
  float* C = nullptr;           // [M][ldc] f32
  long ldc = 0;
  int epi = EPI_BIAS;           // Epi
  // EPI_BIAS_GELU with P set: the result goes to the pair matrix P [M][N]
  // scaled by p_scale[n] instead of C
  uint16_t* P = nullptr;
  const float* p_scale = nullptr;
  // kv.k set (c_attn): the k / v columns of row s * kv_T + t go into the cache
  // at position kv_past + t instead of C
  KvDst kv{};
  int kv_T = 1, kv_past = 0;
  float* ws = nullptr;          // split-k partials
  size_t ws_floats = 0;
};

// Workspace floats launch_pair_gemm uses to split an M x N x K GEMM over k (0:
// it runs unsplit); at most those of the next multiple of 32 rows.
size_t pair_gemm_ws_floats(int M, int N, int K, int planes);
void launch_pair_gemm(hipStream_t s, const PairWeights& w, const PairGemmArgs& a);

}  // namespace rtg
