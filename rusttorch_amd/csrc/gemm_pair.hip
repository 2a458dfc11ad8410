// Prefill GEMM C = epi(A W^T) with f32 operands on f16 MFMA.
//
// CDNA4's f32 MFMA runs at 1/16 of its f16 rate. Here every operand is a pair
// of f16, hi + lo, scaled by powers of two (f16_pair.h), and a product is
// hi hi + hi lo + lo hi: three f16 MFMAs per f32 product, each exact in the
// f32 accumulator's input (11 x 11 bits), so the rounding left is the pair's
// own (2^-24 of a value in the mean, 2^-23 at worst; the dropped lo lo 2^-24 and
// 2^-22 of a product) and the accumulator's, which takes 16
// products per rounding instead of 2. bf16 weights fit one f16: two MFMAs.
// The scales are fixed when the model is loaded, from bounds that hold for
// every input (gemm_pair.h), so no value overflows f16.
//
// What bounds it: at 16368 x 5120 x 1280 the 256 x 256 tile runs at 378-385
// TFLOP/s of f32 products, 1.15 PFLOP/s of f16 MFMA, what a library f16 GEMM
// reaches on this card (8192^3: 1.09); the f32-MFMA kernel runs at
// 126 (157 peak) and is further from 64 bits (6.6e-7 against 3.9e-7 relative
// at K = 1280, 1.24e-6 against 8.0e-7 at 5120). At a few hundred rows the
// launch, the first loads and the chain of k-tiles bound it (gemm_pair_choice.h).
//
// A workgroup computes BM x BN outputs from k-tiles of 32: LDS rows of 128
// bytes [32 hi][32 lo] (64 bytes for one-plane weights), filled by LDS-direct
// loads in a ring of NS stages, 16-byte chunks XOR-swizzled so that the 16 lanes
// of an LDS read cycle (consecutive rows) cover its 64 banks: two 128-byte
// rows span them, so the swizzle is row / 2 (row / 4 for 64-byte rows). By the
// row itself every read took twice its cycles (SQ_LDS_BANK_CONFLICT 6.9e7 per
// dispatch of 32768 x 1280 x 3840-5120, now 0): 1.66e7 -> 1.64e7 cycles, the
// 128 x 128 tiles 1.28e7 -> 1.26e7. By the counters the MFMAs are busy half of
// the cycles, at about 1.9 GHz; what takes the other half is not pinned down.
#include "gemm_pair.h"

#include <algorithm>
#include <type_traits>

#include "f16_pair.h"
#include "gelu.h"
#include "gemm_pair_choice.h"

namespace rtg {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// ---- scales and weights, once per model ----

// The power of two that brings a bound below 2^15 (1 for a zero bound), at most
// 2^80. A bound of 2^95 or more (or none) sets *bad: no scale down to 2^-80
// keeps such values in f16.
__device__ __forceinline__ float scale_of(double bound, int* bad) {
  if (!(bound < 0x1p95)) {
    *bad = 1;
    return 1.f;
  }
  if (bound == 0.0) return 1.f;
  int e;
  frexp(bound, &e);  // bound < 2^e <= 2^95
  return (float)ldexp(1.0, min(15 - e, 80));
}

__global__ __launch_bounds__(256) void pair_ln_scale_kernel(const float* __restrict__ g, const float* __restrict__ b,
                                                            int d, float* __restrict__ scale, int* bad) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < d) scale[k] = scale_of(sqrt((double)d) * fabs((double)g[k]) + fabs((double)b[k]), bad);
}

// Four consecutive weights (i % 4 == 0).
__device__ __forceinline__ float4 weights_at(const void* W, int wtype, size_t i) {
  if (wtype == W_F32) return *reinterpret_cast<const float4*>(static_cast<const float*>(W) + i);
  const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(W) + i);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xffff0000u));
}

__device__ __forceinline__ double wave_sum_d(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ __launch_bounds__(256) void pair_row_scale_kernel(const void* __restrict__ W, int wtype, int N, int K,
                                                             const float* __restrict__ g, const float* __restrict__ b,
                                                             const float* __restrict__ bias,
                                                             float* __restrict__ scale, int* bad) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  double sq = 0.0, c = 0.0;
  auto add = [&](float w, float gk, float bk) {
    const double wg = (double)w * (double)gk;
    sq += wg * wg;
    c += (double)w * (double)bk;
  };
  for (int k = lane * 4; k < K; k += 256) {
    const float4 w = weights_at(W, wtype, (size_t)n * K + k);
    const float4 gk = *reinterpret_cast<const float4*>(g + k), bk = *reinterpret_cast<const float4*>(b + k);
    add(w.x, gk.x, bk.x);
    add(w.y, gk.y, bk.y);
    add(w.z, gk.z, bk.z);
    add(w.w, gk.w, bk.w);
  }
  sq = wave_sum_d(sq);
  c = wave_sum_d(c);
  if (lane == 0) scale[n] = scale_of(sqrt((double)K * sq) + fabs(c + (double)bias[n]), bad);
}

// The k-tiles (of 32) whose weights are stored negated, of a row's nkt: the two
// middle quarters (see pair_gemm_kernel).
__device__ __forceinline__ int flip_begin(int nkt) { return nkt / 4; }
__device__ __forceinline__ int flip_end(int nkt) { return nkt - nkt / 4; }

// One wave per row: the row's largest |W / in_scale|, then the scaled pairs.
// Scales are powers of two, so the products are exact; a row whose largest
// entry is outside [2^-90, 2^90] sets *bad.
__global__ __launch_bounds__(256) void pair_weights_kernel(const void* __restrict__ W, int wtype, int N, int K,
                                                           const float* __restrict__ in_scale, int planes,
                                                           uint16_t* __restrict__ out, float* __restrict__ out_scale,
                                                           int* bad) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  auto load = [&](int k) {
    float4 w = weights_at(W, wtype, (size_t)n * K + k);
    const float4 t = *reinterpret_cast<const float4*>(in_scale + k);
    return make_float4(w.x / t.x, w.y / t.y, w.z / t.z, w.w / t.w);
  };
  float top = 0.f;
  bool fine = true;
  for (int k = lane * 4; k < K; k += 256) {
    const float4 v = load(k);
    const float a[4] = {fabsf(v.x), fabsf(v.y), fabsf(v.z), fabsf(v.w)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      fine = fine && a[i] < INFINITY;  // (false for NaN)
      top = fmaxf(top, a[i]);
    }
  }
  for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
  int e = 0;
  if (top > 0.f) frexpf(top, &e);
  if (!fine || e < -90 || e > 90) *bad = 1;
  e = min(max(e, -90), 90);
  const float r = ldexpf(1.f, 15 - e);
  if (lane == 0) out_scale[n] = ldexpf(1.f, e - 15);
  for (int k = lane * 4; k < K; k += 256) {
    const float4 v = load(k);
    const float f = (k >> 5) >= flip_begin(K >> 5) && (k >> 5) < flip_end(K >> 5) ? -r : r;
    const float4 y = make_float4(v.x * f, v.y * f, v.z * f, v.w * f);
    if (planes == 2)
      pair_store4(out, n, k, K, y);
    else
      *reinterpret_cast<uint2*>(out + (size_t)n * K + k) =
          make_uint2(f16_bits(y.x) | f16_bits(y.y) << 16, f16_bits(y.z) | f16_bits(y.w) << 16);
  }
}

// ---- the GEMM ----

// One LDS-direct load instruction: lane i's 16 bytes at base + voff go to LDS
// lds + 16 i. Written out so that the compiler's wait-count pass does not tie
// the LDS reads of other stages to it; the kernel waits itself.
__device__ __forceinline__ void dma16(unsigned voff, const void* base, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}
// At most N of this wave's loads outstanding and its LDS reads complete, then
// the barrier. (The reads' results may be used behind it: nothing but this wait
// keeps another wave's load from overwriting a stage still being read.)
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ f16x8 lds_frag(const char* p) { return *reinterpret_cast<const f16x8*>(p); }
// v with every element's sign bit flipped where sign is 0x80008000.
__device__ __forceinline__ f16x8 signed_frag(const f16x8& v, unsigned sign) {
  const uint4 u = __builtin_bit_cast(uint4, v);
  return __builtin_bit_cast(f16x8, make_uint4(u.x ^ sign, u.y ^ sign, u.z ^ sign, u.w ^ sign));
}

struct Out {
  const float* bias;
  const float* out_scale;
  float* C;
  long ldc;
  int epi;
  uint16_t* P;
  const float* p_scale;
  KvDst kv;
  int kv_T, kv_past;
  unsigned long long kv_magic;  // ceil(2^40 / kv_T): m / kv_T = m kv_magic >> 40 for m kv_T < 2^40
};

// What becomes of an output column's values (wave-uniform).
enum Put { PUT_RAW, PUT_BIAS, PUT_RESID, PUT_PAIR, PUT_KV };

__device__ __forceinline__ int put_of(const Out& o, int n) {
  if (o.P != nullptr) return PUT_PAIR;
  if (o.kv.k != nullptr && n >= o.kv.d) return PUT_KV;
  return o.epi == EPI_NONE ? PUT_RAW : o.epi == EPI_BIAS_RESID ? PUT_RESID : PUT_BIAS;
}

// Output v (scaled back, no bias) of row m < M, column n. PUT_PAIR: every
// lane of the wave calls it (rows past M are not stored).
template <int PUT>
__device__ __forceinline__ void put(const Out& o, int M, int N, int m, int n, float v, float bv, float ps) {
  if (PUT == PUT_PAIR) {
    // the even lane of a column pair stores both his, the odd lane both los:
    // 4-byte stores, 32 lanes one whole 128-byte group
    unsigned h, l;
    f16_split(gelu_new(v + bv) * ps, &h, &l);
    const bool odd = n & 1;
    const unsigned got =
        (unsigned)__builtin_amdgcn_update_dpp(0, (int)(odd ? h : l), 0xB1, 0xF, 0xF, false);  // of lane ^ 1
    const unsigned word = odd ? got | l << 16 : h | got << 16;
    if (m < M) *reinterpret_cast<unsigned*>(o.P + pair_index((size_t)m, n & ~1, N) + (odd ? 32 : 0)) = word;
    return;
  }
  if (m >= M) return;
  if (PUT == PUT_KV) {
    const int which = n >= 2 * o.kv.d, cc = n - o.kv.d - which * o.kv.d;
    const int hd = o.kv.d / o.kv.n_head, hh = cc / hd;
    const int sq = (int)((unsigned long long)m * o.kv_magic >> 40), t = m - sq * o.kv_T;
    float* base = which ? o.kv.v : o.kv.k;
    base[(((size_t)sq * o.kv.n_head + hh) * o.kv.n_pos + o.kv_past + t) * hd + (cc - hh * hd)] = v + bv;
    return;
  }
  float* cp = o.C + (size_t)m * o.ldc + n;
  if (PUT == PUT_RAW) *cp = v;
  else if (PUT == PUT_BIAS) *cp = v + bv;
  else *cp = *cp + (v + bv);
}

// Signs: an MFMA rounds the small terms of its sum towards minus infinity, so
// cross products accumulated onto a large sum leave every output short by the
// same amount (16368 x 3840 x 1280: 3.1e-8 of its root mean square, 0.077 of the
// error's standard deviation), which an average over a thousand keys keeps while
// it shrinks every other error. The weights of the two middle quarters of k are
// therefore stored negated and the sum changes sign with them: the bias there
// takes back that of the outer quarters (the sums grow like the square root of
// k, so + - - + leaves a twentieth): now below 0.001, for 0.8% of the time (a
// change of sign every 4 k-tiles: 2.6%; operands negated in registers: 6%).
// DUAL's cross products meet small sums only (0.004 without this): those tiles
// take the weights' signs back.
//
// WM x WN waves, each MI x NJ blocks of 32 x 32; PW weight planes; NS stages.
// KW = 2: twice the waves, each pair sharing its blocks and taking one half
// of every k-tile. DUAL: the cross products hi lo + lo hi have their own
// accumulators (a third of the roundings of the large sum).
template <int PW, int WM, int WN, int MI, int NJ, int NS, int KW>
struct Tile {
  static constexpr int NW = WM * WN * KW, BM = WM * MI * 32, BN = WN * NJ * 32;
  // 1 KiB load instructions of a stage: A groups of 8 rows x 128 bytes, W
  // groups of the same (one plane: 16 rows x 64 bytes), LD per wave
  static constexpr int GA = BM / 8, G = GA + BN * PW / 16, LD = (G + NW - 1) / NW;
  static constexpr int A_BYTES = BM * 128, STAGE = A_BYTES + BN * 64 * PW;
};

template <int PW, int WM, int WN, int MI, int NJ, int NS, int KW, bool DUAL>
__global__ __launch_bounds__(64 * WM * WN * KW) void pair_gemm_kernel(const uint16_t* __restrict__ A, long lda, int M,
                                                                 const uint16_t* __restrict__ W, int N, int K, int ks,
                                                                 int gm, Out out, float* __restrict__ ws) {
  using T = Tile<PW, WM, WN, MI, NJ, NS, KW>;
  __shared__ __attribute__((aligned(128))) char lds[NS * T::STAGE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block order: workgroups go to the 8 XCDs in turn, so each XCD takes a
  // contiguous range of tiles, ordered in groups of gm row blocks by columns,
  // whose operands its L2 holds.
  const int nmb = (M + T::BM - 1) / T::BM, nnb = (N + T::BN - 1) / T::BN, tiles = nmb * nnb, total = tiles * ks;
  int t = blockIdx.x;
  {
    const int x = t & 7, q = total >> 3, r = total & 7;
    t = x * q + min(x, r) + (t >> 3);
  }
  const int z = t / tiles;
  t -= z * tiles;
  const int wide = gm * nnb, first = t / wide * gm, rows = min(nmb - first, gm), in = t % wide;
  const int m0 = (first + in % rows) * T::BM, n0 = in / rows * T::BN;
  const int nk = K / 32 / ks;  // k-tiles of this split

  // This wave's loads: groups wave * LD + q (past the last: the last again, so
  // that every wave has LD in flight per stage), as byte offsets from the
  // tile's first row at this split's first k; the lane's chunk is the
  // swizzled one.
  const char* abase = reinterpret_cast<const char*>(A + (size_t)m0 * lda) + (size_t)z * nk * 128;
  const char* wbase = reinterpret_cast<const char*>(W + (size_t)n0 * K * PW) + (size_t)z * nk * 64 * PW;
  unsigned off[T::LD];
#pragma unroll
  for (int q = 0; q < T::LD; ++q) {
    const int g = min(wave * T::LD + q, T::G - 1);
    const int swz = (g & 1) << 2 | lane >> 4;  // (row / 2) % 8 of row 8 g + lane / 8 (GA is even)
    if (g < T::GA)
      off[q] = (unsigned)min(g * 8 + (lane >> 3), M - 1 - m0) * (unsigned)(lda * 2) + (((lane & 7) ^ swz) << 4);
    else if (PW == 2)
      off[q] = (unsigned)min((g - T::GA) * 8 + (lane >> 3), N - 1 - n0) * (unsigned)(K * 4) +
               (((lane & 7) ^ swz) << 4);
    else
      off[q] = (unsigned)min((g - T::GA) * 16 + (lane >> 2), N - 1 - n0) * (unsigned)(K * 2) +
               (((lane & 3) ^ (lane >> 4)) << 4);
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  auto issue = [&](int kt, int st) {
    const char* ap = abase + (size_t)kt * 128;
    const char* wp = wbase + (size_t)kt * 64 * PW;
#pragma unroll
    for (int q = 0; q < T::LD; ++q) {
      const int g = min(wave * T::LD + q, T::G - 1);
      dma16(off[q], g < T::GA ? ap : wp, __builtin_amdgcn_readfirstlane(lds0 + st * T::STAGE + g * 1024));
    }
  };

  // operand reads: row lane % 32 of a 32-row block, k half lane / 32: chunk
  // plane * 4 + step * 2 + half (one plane: step * 2 + half), swizzled
  const int kz = wave / (WM * WN), wt = wave % (WM * WN);
  const int wm = wt / WN * MI * 32, wn = wt % WN * NJ * 32, h = lane >> 5, r31 = lane & 31;
  int ard[2][2], wrd[PW][2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int s = 0; s < 2; ++s) ard[p][s] = (wm + r31) * 128 + (((p * 4 + s * 2 + h) ^ ((lane >> 1) & 7)) << 4);
#pragma unroll
  for (int p = 0; p < PW; ++p)
#pragma unroll
    for (int s = 0; s < 2; ++s)
      wrd[p][s] = T::A_BYTES + (PW == 2 ? (wn + r31) * 128 + (((p * 4 + s * 2 + h) ^ ((lane >> 1) & 7)) << 4)
                                        : (wn + r31) * 64 + (((s * 2 + h) ^ ((lane >> 2) & 3)) << 4));

  int arz[2], wrz[PW];  // those of this wave's half (KW = 2)
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    arz[p] = kz ? ard[p][1] : ard[p][0];
    if (p < PW) wrz[p] = kz ? wrd[p][1] : wrd[p][0];
  }

  floatx16 acc[MI][NJ], acx[DUAL ? MI : 1][DUAL ? NJ : 1];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][j][e] = 0.f;
        if (DUAL) acx[i][j][e] = 0.f;
      }

#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < nk) issue(p, p);
  auto negate = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc[i][j][e] = -acc[i][j][e];
        }
  };
  const int kt0 = z * nk, neg0 = flip_begin(K / 32) - kt0, neg1 = flip_end(K / 32) - kt0;
  int st = 0;
  auto tile = [&](int kt) {
    // tile kt has landed once only the loads of the NS - 2 later tiles are
    // outstanding; past the barrier that holds for every wave, and no wave
    // reads the stage that is filled next any more
    if (kt + NS - 2 < nk) wait_barrier<(NS - 2) * T::LD>();
    else wait_barrier<0>();
    if (kt + NS - 1 < nk) issue(kt + NS - 1, st == 0 ? NS - 1 : st - 1);
    const char* sp = lds + st * T::STAGE;
    const unsigned sign = DUAL && kt >= neg0 && kt < neg1 ? 0x80008000u : 0u;
#pragma unroll
    for (int s0 = 0; s0 < 2; s0 += KW) {
      const int s = KW == 2 ? kz : s0;
      f16x8 a[2][MI], w[PW][NJ];
#pragma unroll
      for (int p = 0; p < PW; ++p)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          w[p][j] = lds_frag(sp + (KW == 2 ? wrz[p] : wrd[p][s0]) + j * 32 * 64 * PW);
          if (DUAL) w[p][j] = signed_frag(w[p][j], sign);
        }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < MI; ++i) a[p][i] = lds_frag(sp + (KW == 2 ? arz[p] : ard[p][s0]) + i * 32 * 128);
      (void)s;
      auto mma = [&](const f16x8 (&x)[MI], const f16x8 (&y)[NJ], auto& to) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i], y[j], to[i][j], 0, 0, 0);
      };
      if constexpr (DUAL) {
        mma(a[1], w[0], acx);
        mma(a[0], w[0], acc);
        if (PW == 2) mma(a[0], w[PW - 1], acx);
      } else {
        mma(a[1], w[0], acc);
        if (PW == 2) mma(a[0], w[PW - 1], acc);
        mma(a[0], w[0], acc);
      }
    }
    st = st + 1 == NS ? 0 : st + 1;
  };
  if constexpr (DUAL) {
    for (int kt = 0; kt < nk; ++kt) tile(kt);
  } else {
    // the three runs of equal sign, as far as this split has k-tiles of them
    int kt = 0;
#pragma unroll 1
    for (int run = 0; run < 3; ++run) {
      const int end = run == 2 ? nk : min(nk, run == 0 ? neg0 : neg1);
      for (; kt < end; ++kt) tile(kt);
      if (run < 2) negate();
    }
  }

  if constexpr (DUAL) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += acx[i][j][e];
  }
  if constexpr (KW == 2) {
    // the second half's sums join the first's through LDS
    float* red = reinterpret_cast<float*>(lds) + (size_t)wt * (MI * NJ * 16 * 64) + lane;
    __syncthreads();  // every wave is done with the stages
    if (kz == 1) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) red[((i * NJ + j) * 16 + e) * 64] = acc[i][j][e];
    }
    __syncthreads();
    if (kz == 1) return;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += red[((i * NJ + j) * 16 + e) * 64];
  }

  // lane holds D[(e / 4) * 8 + h * 4 + e % 4][r31] of each block in acc[e]
  auto column = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    const int n = n0 + wn + j * 32 + r31;
    if (n >= N) return;
    const float sc = out.out_scale[n], bv = out.bias ? out.bias[n] : 0.f, ps = out.P ? out.p_scale[n] : 1.f;
    auto each = [&](auto&& f) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) f(m0 + wm + i * 32 + (e >> 2) * 8 + h * 4 + (e & 3), acc[i][j][e]);
    };
    if (ws != nullptr) {
      each([&](int m, float v) {
        if (m < M) ws[((size_t)z * M + m) * N + n] = v;
      });
      return;
    }
    switch (put_of(out, n0 + wn + j * 32)) {
      case PUT_RAW: each([&](int m, float v) { put<PUT_RAW>(out, M, N, m, n, v * sc, bv, ps); }); break;
      case PUT_BIAS: each([&](int m, float v) { put<PUT_BIAS>(out, M, N, m, n, v * sc, bv, ps); }); break;
      case PUT_RESID: each([&](int m, float v) { put<PUT_RESID>(out, M, N, m, n, v * sc, bv, ps); }); break;
      case PUT_PAIR: each([&](int m, float v) { put<PUT_PAIR>(out, M, N, m, n, v * sc, bv, ps); }); break;
      default: each([&](int m, float v) { put<PUT_KV>(out, M, N, m, n, v * sc, bv, ps); }); break;
    }
  };
  column(std::integral_constant<int, 0>{});
  if constexpr (NJ > 1) column(std::integral_constant<int, 1>{});
  static_assert(NJ <= 2, "columns of blocks");
}

// Sum of the ks split-k partials (in split order) and the epilogue.
__global__ __launch_bounds__(256) void pair_reduce_kernel(const float* __restrict__ ws, int ks, int M, int N,
                                                          Out out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const size_t MN = (size_t)M * N;
  if (i >= (long)MN) return;
  const int m = (int)(i / N), n = (int)(i - (long)m * N);
  float t[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) t[u] = u < ks ? ws[(size_t)u * MN + i] : 0.f;
  float v = t[0];
#pragma unroll
  for (int u = 1; u < 16; ++u)
    if (u < ks) v += t[u];
  v *= out.out_scale[n];
  const float bv = out.bias ? out.bias[n] : 0.f, ps = out.P ? out.p_scale[n] : 1.f;
  switch (put_of(out, n)) {
    case PUT_RAW: put<PUT_RAW>(out, M, N, m, n, v, bv, ps); break;
    case PUT_BIAS: put<PUT_BIAS>(out, M, N, m, n, v, bv, ps); break;
    case PUT_RESID: put<PUT_RESID>(out, M, N, m, n, v, bv, ps); break;
    case PUT_PAIR: put<PUT_PAIR>(out, M, N, m, n, v, bv, ps); break;
    default: put<PUT_KV>(out, M, N, m, n, v, bv, ps); break;
  }
}

constexpr int kGroupRows = 8;  // row blocks per group of the block order (4 and 16 measured the same)

template <int PW, int WM, int WN, int MI, int NJ, int NS, int KW = 1, bool DUAL = false>
void launch_tile(hipStream_t s, const PairWeights& w, const PairGemmArgs& a, int ks) {
  using T = Tile<PW, WM, WN, MI, NJ, NS, KW>;
  static_assert(NS * T::STAGE <= 160 * 1024 && (KW == 1 || T::BM * T::BN * 4 <= NS * T::STAGE), "LDS");
  const int tiles = ((a.M + T::BM - 1) / T::BM) * ((w.N + T::BN - 1) / T::BN);
  const Out o{a.bias, w.out_scale, a.C, a.ldc, a.epi, a.P, a.p_scale, a.kv, a.kv_T, a.kv_past,
              ((1ull << 40) + a.kv_T - 1) / a.kv_T};
  pair_gemm_kernel<PW, WM, WN, MI, NJ, NS, KW, DUAL><<<tiles * ks, T::NW * 64, 0, s>>>(
      a.A, a.lda, a.M, w.w, w.N, w.K, ks, kGroupRows, o, ks > 1 ? a.ws : nullptr);
  if (ks > 1)
    pair_reduce_kernel<<<(unsigned)(((long)a.M * w.N + 255) / 256), 256, 0, s>>>(a.ws, ks, a.M, w.N, o);
}

template <int PW>
void launch_planes(hipStream_t s, const PairWeights& w, const PairGemmArgs& a) {
  const PairChoice c = pair_choose(a.M, w.N, w.K, PW, a.ws ? a.ws_floats : 0);
  switch (c.tile) {
    case 0: launch_tile<PW, 2, 4, 4, 2, 2>(s, w, a, c.ks); break;
    case 1: launch_tile<PW, 2, 2, 2, 2, 2>(s, w, a, c.ks); break;
    case 2: launch_tile<PW, 2, 4, 2, 1, 3, 1, true>(s, w, a, c.ks); break;
    case 3: launch_tile<PW, 1, 4, 2, 1, 3, 1, true>(s, w, a, c.ks); break;
    case 4: launch_tile<PW, 2, 2, 1, 1, 4, 2, true>(s, w, a, c.ks); break;
    default: launch_tile<PW, 1, 2, 1, 1, 6, 2, true>(s, w, a, c.ks); break;
  }
}

}  // namespace

size_t pair_weight_bytes(int N, int K, int wtype) { return (size_t)N * K * (wtype == W_F32 ? 4 : 2); }

void launch_pair_ln_scale(hipStream_t s, const float* g, const float* b, int d, float* scale, int* bad) {
  pair_ln_scale_kernel<<<(d + 255) / 256, 256, 0, s>>>(g, b, d, scale, bad);
}
void launch_pair_row_scale(hipStream_t s, const void* W, int wtype, int N, int K, const float* g, const float* b,
                           const float* bias, float* scale, int* bad) {
  pair_row_scale_kernel<<<(N + 3) / 4, 256, 0, s>>>(W, wtype, N, K, g, b, bias, scale, bad);
}
void launch_pair_weights(hipStream_t s, const void* W, int wtype, const float* in_scale, const PairWeights& pw,
                         int* bad) {
  pair_weights_kernel<<<(pw.N + 3) / 4, 256, 0, s>>>(W, wtype, pw.N, pw.K, in_scale, pw.planes, pw.w, pw.out_scale,
                                                    bad);
}

size_t pair_gemm_ws_floats(int M, int N, int K, int planes) {
  const int ks = pair_choose(M, N, K, planes, kSplitMaxFloats).ks;
  return ks > 1 ? (size_t)ks * M * N : 0;
}

void launch_pair_gemm(hipStream_t s, const PairWeights& w, const PairGemmArgs& a) {
  if (w.planes == 2) launch_planes<2>(s, w, a);
  else launch_planes<1>(s, w, a);
}

}  // namespace rtg
