// Prefill causal attention for head_dim 64 on f16 MFMA over f16 pairs
// (flash-attention form of multi_head_attention_cached, gpt2.rs:772-834): f32
// products as three f16 products, as in gemm_pair.hip.
//
// A wave owns 32 queries and walks the keys in blocks of 32. Per block it
// computes S^T = K Q^T (32 keys x 32 queries: v_mfma_f32_32x32x16_f16 over four
// steps of 16 dims), so accumulator i of lane l holds the score of query l % 32
// with key r(i, l) = (i / 4) * 8 + (l / 32) * 4 + i % 4; softmax statistics are
// lane-local plus one exchange between the lane halves. O^T += V^T P^T runs per
// 32-dim tile over two steps of 16 keys; the keys of a step are numbered so
// that the eight a lane half contributes, (t, h, e) -> 16 t + 8 (e / 4) + 4 h +
// e % 4, are the lane's own accumulators 8 t .. 8 t + 7: P feeds the MFMA from
// registers. The running maximum, the sums and O are f32.
//
// Operands: q, k and v scaled per column (the scales of c_attn's outputs, fixed
// when the model is loaded; a head's k scales such that the product with q's is
// the same in every column), P by 2^14; V's scale is the
// attention output's own, so O / (2^14 l) is the pair GEMM's input as it is.
// K and V are read from the f32 cache and split while a block is staged in LDS:
// K rows of 64 hi + 64 lo (256 bytes), V^T rows (one per dim) of 32 hi + 32 lo
// in the key order above (128 bytes), 16-byte chunks XOR-swizzled so that the 16
// lanes of an LDS read cycle cover its 64 banks (K by row % 16: by row % 8 its
// reads took twice their cycles, 6.20e6 against 6.08e6 in all at 32 x 1024).
//
// What bounds it: the vector work around the MFMAs (masks, exponentials,
// splitting P, K and V), about 1250 cycles per block and wave against 768 of
// MFMA. 16 x 1023 tokens, 20 heads: 206 us per layer (165 TFLOP/s) where the f32
// MFMA form, bound by its 4096 MFMA cycles per block, took 541; 701 tokens, 16
// heads (keys split over 8 waves): 21 us against 25; 24 x 50 tokens, 12 heads:
// 12 us against 21. Waves skip key blocks past their own last query.
#include "attn_pair.h"

#include "attn_core.h"
#include "f16_pair.h"

namespace rtg {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int AP_Q = 32;          // queries per wave
constexpr int AP_K = 32;          // keys per block
constexpr int AP_KB = 32 * 256;   // LDS bytes of a K block
constexpr int AP_VB = 64 * 128;   // of a V^T block
constexpr float AP_PS = 16384.f;  // scale of P

// (v0, v1) * s as packed pairs.
__device__ __forceinline__ void split2(float v0, float v1, unsigned* hi, unsigned* lo) {
  const f16x2 h = {(_Float16)v0, (_Float16)v1};
  const f16x2 l = {(_Float16)(v0 - (float)h[0]), (_Float16)(v1 - (float)h[1])};
  *hi = __builtin_bit_cast(unsigned, h);
  *lo = __builtin_bit_cast(unsigned, l);
}

__device__ __forceinline__ int v_swz(int dim) { return (dim ^ (dim >> 3)) & 7; }

// One block's rows of one thread: item e = tid + u NT of 256 is keys 2 (e / 16)
// and the next, dims 4 (e % 16) .. + 3 (rows past kmax are zero).
template <int NT, int U>
struct Stage {
  float4 k[U][2], v[U][2];
  __device__ __forceinline__ void load(const float* Kh, const float* Vh, int kb, int kmax, int tid) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = tid + u * NT;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int j = kb * AP_K + 2 * (e >> 4) + r;
        const size_t at = (size_t)j * 64 + (e & 15) * 4;
        k[u][r] = j <= kmax ? *reinterpret_cast<const float4*>(Kh + at) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[u][r] = j <= kmax ? *reinterpret_cast<const float4*>(Vh + at) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  }
  __device__ __forceinline__ void store(char* Ks, char* Vt, const float4& ak, const float4& av, int tid) const {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = tid + u * NT, key = 2 * (e >> 4), d4 = (e & 15) * 4;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int row = key + r;
        uint2 h, l;
        split2(k[u][r].x * ak.x, k[u][r].y * ak.y, &h.x, &l.x);
        split2(k[u][r].z * ak.z, k[u][r].w * ak.w, &h.y, &l.y);
        char* p = Ks + row * 256 + (d4 & 4) * 2;
        *reinterpret_cast<uint2*>(p + (((d4 >> 3) ^ (row & 15)) << 4)) = h;
        *reinterpret_cast<uint2*>(p + (((8 + (d4 >> 3)) ^ (row & 15)) << 4)) = l;
      }
      // V^T: the key pair's word in chunk (t, half) of four dims' rows
      const int c = (key >> 4) * 2 + ((key >> 2) & 1), in = ((key >> 3) & 1) * 8 + (key & 3) * 2;
      const float a[4] = {v[u][0].x * av.x, v[u][0].y * av.y, v[u][0].z * av.z, v[u][0].w * av.w};
      const float b[4] = {v[u][1].x * av.x, v[u][1].y * av.y, v[u][1].z * av.z, v[u][1].w * av.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        unsigned h, l;
        split2(a[i], b[i], &h, &l);
        const int dim = d4 + i;
        char* p = Vt + dim * 128 + in;
        *reinterpret_cast<unsigned*>(p + ((c ^ v_swz(dim)) << 4)) = h;
        *reinterpret_cast<unsigned*>(p + (((4 + c) ^ v_swz(dim)) << 4)) = l;
      }
    }
  }
};

// A wave's queries and running softmax state.
struct State {
  f16x8 qh[4], ql[4];
  floatx16 o0, o1;
  float m, l;
  __device__ __forceinline__ void init(const float* qrow, const float* aq, int hh) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float4 a = *reinterpret_cast<const float4*>(qrow + 16 * s + 8 * hh);
      const float4 b = *reinterpret_cast<const float4*>(qrow + 16 * s + 8 * hh + 4);
      const float4 sa = *reinterpret_cast<const float4*>(aq + 16 * s + 8 * hh);
      const float4 sb = *reinterpret_cast<const float4*>(aq + 16 * s + 8 * hh + 4);
      unsigned h[4], l4[4];
      split2(a.x * sa.x, a.y * sa.y, &h[0], &l4[0]);
      split2(a.z * sa.z, a.w * sa.w, &h[1], &l4[1]);
      split2(b.x * sb.x, b.y * sb.y, &h[2], &l4[2]);
      split2(b.z * sb.z, b.w * sb.w, &h[3], &l4[3]);
      qh[s] = __builtin_bit_cast(f16x8, make_uint4(h[0], h[1], h[2], h[3]));
      ql[s] = __builtin_bit_cast(f16x8, make_uint4(l4[0], l4[1], l4[2], l4[3]));
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) o0[i] = o1[i] = 0.f;
    m = -INFINITY;
    l = 0.f;
  }
  // Key block j0 .. j0 + 31; fac: score of the scaled dot product, in exp2 units.
  __device__ __forceinline__ void block(const char* Ks, const char* Vt, int j0, int qpos, float fac, int c, int hh) {
    floatx16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const char* row = Ks + c * 256;
      const f16x8 kh = *reinterpret_cast<const f16x8*>(row + (((2 * st + hh) ^ (c & 15)) << 4));
      const f16x8 kl = *reinterpret_cast<const f16x8*>(row + (((8 + 2 * st + hh) ^ (c & 15)) << 4));
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[st], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[st], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[st], s, 0, 0, 0);
    }
    // causal mask (key j <= query position) and online softmax, the scores in
    // units of log2 e (exp(x) = 2^(x log2 e))
    float bm = -INFINITY;
    if (j0 + AP_K - 1 > qpos) {  // (per lane: only blocks that reach past some query)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (j0 + (i >> 2) * 8 + hh * 4 + (i & 3) > qpos) s[i] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) bm = fmaxf(bm, s[i]);
    bm = xor32_max_k(bm) * fac;
    const float mn = fmaxf(m, bm);
    const float corr = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
    const float base = mn == -INFINITY ? 0.f : mn;  // (no key of this query yet: every p is 2^-inf = 0)
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], fac, -base));
      ps += s[i];
    }
    l = l * corr + ps;
    m = mn;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      o0[i] *= corr;
      o1[i] *= corr;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      unsigned h[4], lo[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split2(s[8 * t + 2 * e] * AP_PS, s[8 * t + 2 * e + 1] * AP_PS, &h[e], &lo[e]);
      const f16x8 ph = __builtin_bit_cast(f16x8, make_uint4(h[0], h[1], h[2], h[3]));
      const f16x8 pl = __builtin_bit_cast(f16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int dim = 32 * d + c;
        const char* row = Vt + dim * 128;
        const f16x8 vh = *reinterpret_cast<const f16x8*>(row + (((2 * t + hh) ^ v_swz(dim)) << 4));
        const f16x8 vl = *reinterpret_cast<const f16x8*>(row + (((4 + 2 * t + hh) ^ v_swz(dim)) << 4));
        floatx16& o = d ? o1 : o0;
        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph, o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl, o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph, o, 0, 0, 0);
      }
    }
  }
};

// score = (K . Q) / 8 (1 / sqrt(64)), in units of log2 e, of the scaled operands;
// finite and not zero (head_scale_kernel), so that a masked score stays -inf
__device__ __forceinline__ float score_factor(float qk) { return 0.125f * 1.4426950408889634f / qk; }

// FW waves, each with its own 32 queries of one (sequence, head), over the
// same key blocks: the next block's rows are loaded while this one is used.
template <int FW>
__global__ __launch_bounds__(64 * FW, 2) void attn_pair_kernel(const float* __restrict__ qkv, int T, int past,
                                                            const float* __restrict__ kc,
                                                            const float* __restrict__ vc, int H, int P, int d,
                                                            int nqb, AttnScales sc, uint16_t* __restrict__ out) {
  constexpr int NT = 64 * FW, U = 256 / NT;
  __shared__ __attribute__((aligned(16))) char Ks[AP_KB], Vt[AP_VB];
  // the query block is the slowest grid dimension, longest (last) blocks
  // first: every (sequence, head)'s longest block is dispatched before any
  // shorter one, which keeps the tail of the grid short
  const int qb = nqb - 1 - (int)blockIdx.z;
  const int h = blockIdx.x, sidx = blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 31, hh = lane >> 5;
  const int qi = qb * AP_Q * FW + wave * AP_Q + c;  // this lane's query
  const int qpos = past + qi;
  const size_t head_off = ((size_t)sidx * H + h) * (size_t)P * 64;
  const float *Kh = kc + head_off, *Vh = vc + head_off;
  const float4 ak = *reinterpret_cast<const float4*>(sc.k + h * 64 + (tid & 15) * 4);
  const float4 av = *reinterpret_cast<const float4*>(sc.v + h * 64 + (tid & 15) * 4);
  const float fac = score_factor(sc.qk[h]);
  const int kmax = past + min(T, (qb + 1) * AP_Q * FW) - 1;  // last key any query here attends
  const int nkb = kmax / AP_K + 1;
  // (a wave past its own last key block only stages: its queries are earlier)
  const int mine = (past + min(T, qb * AP_Q * FW + (wave + 1) * AP_Q) - 1) / AP_K + 1;
  Stage<NT, U> st;
  st.load(Kh, Vh, 0, kmax, tid);
  State q;
  q.init(qkv + ((size_t)sidx * T + min(qi, T - 1)) * 3 * d + h * 64, sc.q + h * 64, hh);
  for (int kb = 0; kb < nkb; ++kb) {
    __syncthreads();  // every wave is done with the previous block
    st.store(Ks, Vt, ak, av, tid);
    __syncthreads();
    if (kb + 1 < nkb) st.load(Kh, Vh, kb + 1, kmax, tid);
    if (kb < mine) q.block(Ks, Vt, kb * AP_K, qpos, fac, c, hh);
  }
  const float inv = 1.0f / (AP_PS * xor32_sum_k(q.l));
  if (qi < T) {
    const size_t row = (size_t)sidx * T + qi;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int col = h * 64 + 8 * g + 4 * hh;
      pair_store4(out, row, col, d,
                  make_float4(q.o0[4 * g] * inv, q.o0[4 * g + 1] * inv, q.o0[4 * g + 2] * inv, q.o0[4 * g + 3] * inv));
      pair_store4(out, row, col + 32, d,
                  make_float4(q.o1[4 * g] * inv, q.o1[4 * g + 1] * inv, q.o1[4 * g + 2] * inv, q.o1[4 * g + 3] * inv));
    }
  }
}

// The key range split over KS waves: all have the same 32 queries, wave w
// takes key blocks w, w + KS, ..., each staged in the wave's own LDS region
// (no workgroup barrier per block); the waves' (m, l, O) merge in LDS. For a few
// long prompts the causal chain of the last query block would otherwise be the
// whole kernel.
template <int KS>
__global__ __launch_bounds__(64 * KS, 2) void attn_pair_ks_kernel(const float* __restrict__ qkv, int T, int past,
                                                               const float* __restrict__ kc,
                                                               const float* __restrict__ vc, int H, int P, int d,
                                                               int nqb, AttnScales sc, uint16_t* __restrict__ out) {
  constexpr int MW = 64 + 2;  // merge record of one query: m, l, O[64]
  static_assert(AP_Q * MW * 4 <= AP_KB + AP_VB, "merge records fit the staging region");
  __shared__ __attribute__((aligned(16))) char sm[KS][AP_KB + AP_VB];
  const int qb = nqb - 1 - (int)blockIdx.z;  // longest query blocks first
  const int h = blockIdx.x, sidx = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 31, hh = lane >> 5;
  const int qi = qb * AP_Q + c;
  const int qpos = past + qi;
  const size_t head_off = ((size_t)sidx * H + h) * (size_t)P * 64;
  const float *Kh = kc + head_off, *Vh = vc + head_off;
  char *Ks = sm[wave], *Vt = sm[wave] + AP_KB;
  const float4 ak = *reinterpret_cast<const float4*>(sc.k + h * 64 + (lane & 15) * 4);
  const float4 av = *reinterpret_cast<const float4*>(sc.v + h * 64 + (lane & 15) * 4);
  const float fac = score_factor(sc.qk[h]);
  const int kmax = past + min(T, (qb + 1) * AP_Q) - 1;
  const int nkb = kmax / AP_K + 1;
  Stage<64, 4> st;
  if (wave < nkb) st.load(Kh, Vh, wave, kmax, lane);
  State q;
  q.init(qkv + ((size_t)sidx * T + min(qi, T - 1)) * 3 * d + h * 64, sc.q + h * 64, hh);
  for (int kb = wave; kb < nkb; kb += KS) {
    // this wave's region only: LDS accesses of one wave are ordered, the
    // wave's previous reads are complete before its writes below
    st.store(Ks, Vt, ak, av, lane);
    if (kb + KS < nkb) st.load(Kh, Vh, kb + KS, kmax, lane);
    q.block(Ks, Vt, kb * AP_K, qpos, fac, c, hh);
  }
  const float l = xor32_sum_k(q.l);
  __syncthreads();  // every wave is done with its staging region
  float* rec = reinterpret_cast<float*>(sm[wave]) + c * MW;
  if (hh == 0) {
    rec[0] = q.m;
    rec[1] = l;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = (i / 4) * 8 + hh * 4 + (i % 4);
    rec[2 + r] = q.o0[i];
    rec[2 + 32 + r] = q.o1[i];
  }
  __syncthreads();
  // wave 0 lane (c, hh) merges the 32 dims it holds for query c
  if (wave == 0 && qi < T) {
    auto part = [&](int w) { return reinterpret_cast<const float*>(sm[w]) + c * MW; };
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < KS; ++w) M = fmaxf(M, part(w)[0]);
    float L = 0.f, f[KS];
#pragma unroll
    for (int w = 0; w < KS; ++w) {
      const float mw = part(w)[0];
      f[w] = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
      L += part(w)[1] * f[w];
    }
    const float inv = 1.0f / (AP_PS * L);
    const size_t row = (size_t)sidx * T + qi;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const int r = (g & 3) * 8 + hh * 4 + (g >> 2) * 32;  // four consecutive dims
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < KS; ++w) {
        const float* p = part(w) + 2 + r;
        a.x += p[0] * f[w];
        a.y += p[1] * f[w];
        a.z += p[2] * f[w];
        a.w += p[3] * f[w];
      }
      pair_store4(out, row, h * 64 + r, d, make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv));
    }
  }
}

// A head's k scales and the product qk: the smallest product of a column's q
// and k scales. A column's k scale is then qk over its q scale, at most its own;
// what a column of smaller products loses by that is as far below the head's
// scores as f32's own rounding of them. (One scale for a head's q and one for
// its k lost 2^-15 of every column beside one that is 2^20 larger.)
// Above 2^110 the head's scores are below 2^-77 (64 products of 2^30 over 2^110,
// over 8) and the softmax is uniform whatever they are; a smaller qk keeps the
// score factor from becoming 0, whose product with a masked score is NaN. A
// product below 2^-100 (scores that may pass f32's range) is left to the f32
// attention.
__global__ __launch_bounds__(64) void head_scale_kernel(const float* __restrict__ col, int H, float* __restrict__ k,
                                                        float* __restrict__ qk, int* bad) {
  const int h = blockIdx.x, c = h * 64 + threadIdx.x;
  const int eq = ilogbf(col[c]), e = eq + ilogbf(col[H * 64 + c]);
  int least = e;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) least = min(least, __shfl_xor(least, o, 64));
  if (least < -100) *bad = 1;
  least = min(least, 110);
  k[c] = ldexpf(1.f, least - eq);
  if (threadIdx.x == 0) qk[h] = ldexpf(1.f, least);
}

}  // namespace

void launch_head_scale(hipStream_t s, const float* col, int H, float* k, float* qk, int* bad) {
  head_scale_kernel<<<H, 64, 0, s>>>(col, H, k, qk, bad);
}

void launch_attn_pair(hipStream_t s, const float* qkv, int S, int T, int past, const float* kc, const float* vc,
                      int n_head, int n_pos, int d, const AttnScales& sc, uint16_t* out) {
  if ((long)n_head * S < 256 && T + past >= 4 * AP_K) {
    // few (sequence, head) pairs with long key ranges: split the keys over 4
    // waves, 8 from 16 key blocks on
    const int nqb = (T + AP_Q - 1) / AP_Q;
    const dim3 grid(n_head, S, nqb);
    if (T + past >= 16 * AP_K)
      attn_pair_ks_kernel<8><<<grid, 512, 0, s>>>(qkv, T, past, kc, vc, n_head, n_pos, d, nqb, sc, out);
    else
      attn_pair_ks_kernel<4><<<grid, 256, 0, s>>>(qkv, T, past, kc, vc, n_head, n_pos, d, nqb, sc, out);
    return;
  }
  // 128 queries per workgroup where that gives two workgroups per CU, else 64
  // or 32 (a short batch of prompts would otherwise leave most CUs idle)
  int fw = 4;
  while (fw > 1 && (long)n_head * S * ((T + AP_Q * fw - 1) / (AP_Q * fw)) < 512) fw >>= 1;
  const int nqb = (T + AP_Q * fw - 1) / (AP_Q * fw);
  const dim3 grid(n_head, S, nqb);
  if (fw == 4)
    attn_pair_kernel<4><<<grid, 256, 0, s>>>(qkv, T, past, kc, vc, n_head, n_pos, d, nqb, sc, out);
  else if (fw == 2)
    attn_pair_kernel<2><<<grid, 128, 0, s>>>(qkv, T, past, kc, vc, n_head, n_pos, d, nqb, sc, out);
  else
    attn_pair_kernel<1><<<grid, 64, 0, s>>>(qkv, T, past, kc, vc, n_head, n_pos, d, nqb, sc, out);
}

}  // namespace rtg
