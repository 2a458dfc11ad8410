// Token choice on the device: sample_logits (rusttorch-core/src/nn/gpt2.rs:
// 871-906) with repetition penalty (:909-921), temperature, top-k (:924-935),
// top-p (:939-970) and sample_from_logits (:973-993); the greedy branch with a
// repetition penalty (:872-880); and sample_with_temperature (:996-1017),
// which is sample_logits without penalty and filters.
//
// The general form (sample_whole): one workgroup of 512 threads per sequence.
// Element i is held in a register
// of thread i % 512 (row i / 512: the row index is the register index, so
// the load is one coalesced sweep and every later pass works on registers).
// The work is VALU-bound on the one CU, so every pass over the row is kept to
// a few instructions per element:
//  - the repetition penalty marks the history in an LDS bitmap and counts it
//    in an LDS hash table; each element tests its bit and, when set, applies
//    the penalty once per occurrence to its register;
//  - top-k and top-p find their cut-off by histogram rounds (radix select).
//    The first round of top-k bins the scaled logits linearly (2048 bins)
//    between their minimum and maximum, the first round of top-p bins the exponent and two
//    mantissa bits of exp(y - max): both spread the values over many bins, so
//    the LDS atomics rarely collide, and both maps are monotone, so the bin of
//    the k-th value (of the mass crossing p) is exact. Later rounds refine the
//    key bits of that bin's members only;
//  - questions in index order (the sampling CDF, the order of top-p ties) are
//    answered from per-(row, wave) partial sums, reduced across the wave by a
//    transposing butterfly (one shuffle per row and stage, halving the rows at
//    each stage).
//
// The uniform draw of generation index g is output number draw0 + g + 1 of
// SplitMix64 seeded with the caller's seed, mix(seed + k * 0x9E3779B97F4A7C15),
// as 24 bits / 2^24: the sequence of the host sampler (the reference draws
// from rand::thread_rng, so its samples are not reproducible at all).
//
// Sums (softmax denominators, top-p masses, the CDF) are formed in a fixed
// order, so results are deterministic, but not in the reference's sequential
// order, and the CDF is compared in unnormalised form (draw * total against
// running sums of exp(y - max)): a draw within rounding distance of a CDF
// boundary can pick the neighbouring token.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "argmax_key.h"
#include "kernels.h"

namespace rtg {
namespace {

constexpr int ST = 512;        // threads (2 waves per SIMD: up to 256 registers each)
constexpr int SW = ST / 64;    // waves
constexpr int MAX_ROWS = 128;  // V <= 65536
constexpr int NB = 2048;       // histogram bins of the widest round (11 bits)
constexpr int PBW = MAX_ROWS * ST / 32;  // words of the token bitmap
constexpr int DMAX = 2048;  // distinct penalised tokens per penalty round
constexpr uint32_t NONE = 0xffffffffu;

__device__ __forceinline__ float wave_max_s(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_min_s(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}

struct SampleSmem {
  float red[2 * SW];
  unsigned wtot[SW];
  union {
    struct {                        // selection and the draw
      unsigned hist[NB];            // counts or fixed-point probability masses per bin
      float seg[MAX_ROWS * SW];     // per (row, wave) values, index order
      float segpre[MAX_ROWS * SW];  // their exclusive prefix sums
    };
    struct {                  // repetition penalty
      uint32_t wordpre[PBW];  // marked tokens in the bitmap words before each word
      uint32_t cnt[DMAX];     // occurrences per marked token, by rank
      float val[DMAX];        // penalised logit per marked token, by rank
    };
  };
  uint32_t pbits[PBW];  // tokens of the history (within the round's range)
  unsigned misc[8];
  unsigned long long key;
  float fmisc[2];
};

// Max / min over the block in a fixed order; every thread gets the result.
__device__ float block_max(float v, SampleSmem& sm) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  v = wave_max_s(v);
  __syncthreads();
  if (l == 0) sm.red[w] = v;
  __syncthreads();
  float t = -INFINITY;
  for (int i = 0; i < SW; ++i) t = fmaxf(t, sm.red[i]);
  return t;
}
__device__ void block_minmax(float& mx, float& mn, SampleSmem& sm) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  mx = wave_max_s(mx);
  mn = wave_min_s(mn);
  __syncthreads();
  if (l == 0) {
    sm.red[w] = mx;
    sm.red[SW + w] = mn;
  }
  __syncthreads();
  mx = -INFINITY;
  mn = INFINITY;
  for (int i = 0; i < SW; ++i) {
    mx = fmaxf(mx, sm.red[i]);
    mn = fminf(mn, sm.red[SW + i]);
  }
}

// Bin of y among NB linear bins from mn (scale bs = (NB - 1) / range, or 0):
// monotone in y; -inf and NaN go to bin 0.
__device__ __forceinline__ unsigned lin_bin(float y, float mn, float bs) {
  return (unsigned)fminf(fmaxf((y - mn) * bs, 0.f), (float)(NB - 1));
}

__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float from_order_key(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Fixed-point probability mass of e (scale ms = 2^31 / sum): rounded to
// nearest, so the error of a sum over many entries stays unbiased (truncation
// would lose half a unit per entry: ~1e-5 over 45k kept entries, enough to
// move the top-p cut).
__device__ __forceinline__ unsigned mass_of(float e, float ms) { return (unsigned)(e * ms + 0.5f); }

__device__ __forceinline__ uint64_t splitmix_at(uint64_t seed, uint64_t k) {
  uint64_t z = seed + k * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Lanes below this one whose bit is set in a wave ballot.
__device__ __forceinline__ int lanes_before(unsigned long long ballot) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ballot >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ballot, 0u));
}

// Exclusive prefix of x over the block in thread order; the total in *total.
__device__ unsigned block_excl_scan(unsigned x, SampleSmem& sm, unsigned* total) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned incl = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  __syncthreads();
  if (lane == 63) sm.wtot[w] = incl;
  __syncthreads();
  unsigned base = 0, tot = 0;
  for (int i = 0; i < SW; ++i) {
    if (i == w) base = tot;
    tot += sm.wtot[i];
  }
  *total = tot;
  return base + incl - x;
}

// Whole block, after the histogram h[NBINS] is complete: the largest bin b
// whose running total from the top, sum_{b' >= b} h[b'], reaches need (>= 1).
// Leaves b (NONE when the bins do not reach need), the total of the bins above
// it and h[b] in misc[0..2]; ends synchronised.
template <int NBINS>
__device__ void block_top_bin(const unsigned* h, unsigned need, SampleSmem& sm) {
  constexpr int BPT = NBINS / ST;
  static_assert(BPT * ST == NBINS, "bins per thread");
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  unsigned v[BPT], s = 0;
#pragma unroll
  for (int k = 0; k < BPT; ++k) {  // thread t: bins NBINS-1-BPT*t-k, descending
    v[k] = h[NBINS - 1 - BPT * t - k];
    s += v[k];
  }
  unsigned incl = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) sm.wtot[w] = incl;
  if (t == 0) sm.misc[0] = NONE;
  __syncthreads();
  unsigned cum = incl - s;
  for (int i = 0; i < w; ++i) cum += sm.wtot[i];
  // running totals only grow: exactly one thread sees need crossed in its bins
  if (cum < need && need <= cum + s) {
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
      if (cum < need && need <= cum + v[k]) {
        sm.misc[0] = (unsigned)(NBINS - 1 - BPT * t - k);
        sm.misc[1] = cum;
        sm.misc[2] = v[k];
      }
      cum += v[k];
    }
  }
  __syncthreads();
}

// A histogram round: hist_begin clears NBINS bins; the caller accumulates;
// hist_end finds the top bin reaching need (results in misc[0..2] for every
// thread).
template <int NBINS>
__device__ __forceinline__ void hist_begin(SampleSmem& sm) {
  for (int b = threadIdx.x; b < NBINS; b += ST) sm.hist[b] = 0u;
  __syncthreads();
}
template <int NBINS>
__device__ __forceinline__ void hist_end(SampleSmem& sm, unsigned need) {
  __syncthreads();
  block_top_bin<NBINS>(sm.hist, need, sm);
}

// Wave 0 only: segpre[i] = sum of seg[0, i) for i < n (n <= 64 * 16), each
// lane summing a contiguous run in order, then the runs' prefix. Returns the
// total to every lane.
__device__ float wave_excl_prefix(const float* seg, float* segpre, int n, int lane) {
  const int per = (n + 63) / 64, b = lane * per, e = min(n, b + per);
  float s = 0.f;
  for (int i = b; i < e; ++i) s += seg[i];
  float incl = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  float run = incl - s;
  for (int i = b; i < e; ++i) {
    segpre[i] = run;
    run += seg[i];
  }
  return __shfl(incl, 63, 64);
}

// One stage of the transposing butterfly over 16-row chunks: N values per
// lane become N/2; the lane with bit O set keeps the upper half.
template <int N, int O>
__device__ __forceinline__ void tr_stage(float (&a)[16], int lane) {
  constexpr int H = N / 2;
  const bool up = (lane & O) != 0;
#pragma unroll
  for (int k = 0; k < H; ++k) {
    const float send = up ? a[k] : a[k + H];
    const float keep = up ? a[k + H] : a[k];
    a[k] = keep + __shfl_xor(send, O, 64);
  }
}

// seg[row * SW + w] = sum of the wave's 64 values of each row (the 64
// consecutive indices row * ST + w * 64 ...). After the four halving stages
// lane l holds row (l >> 2) of its 16-row chunk, summed over its lane group;
// two butterflies finish the sum.
template <int NJ>
__device__ __forceinline__ void seg_sums(const float (&v)[NJ], float* seg, int w, int lane) {
#pragma unroll
  for (int c0 = 0; c0 < NJ; c0 += 16) {
    float a[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) a[k] = c0 + k < NJ ? v[c0 + k] : 0.f;
    tr_stage<16, 32>(a, lane);
    tr_stage<8, 16>(a, lane);
    tr_stage<4, 8>(a, lane);
    tr_stage<2, 4>(a, lane);
    a[0] += __shfl_xor(a[0], 2, 64);
    a[0] += __shfl_xor(a[0], 1, 64);
    const int r = c0 + (lane >> 2);
    if ((lane & 3) == 0 && r < NJ) seg[r * SW + w] = a[0];
  }
}

// Segment sums of v and their prefix (seg, segpre); returns the total.
template <int NJ>
__device__ __forceinline__ float seg_total(const float (&v)[NJ], SampleSmem& sm, int w, int lane) {
  seg_sums<NJ>(v, sm.seg, w, lane);
  __syncthreads();
  if (w == 0) {
    const float tot = wave_excl_prefix(sm.seg, sm.segpre, NJ * SW, lane);
    if (lane == 0) sm.fmisc[1] = tot;
  }
  __syncthreads();
  return sm.fmisc[1];
}

__device__ __forceinline__ uint32_t hist_at(const uint32_t* prompt, int n_prompt, const uint32_t* ids, int q) {
  return q < n_prompt ? prompt[q] : ids[q - n_prompt];
}

// Dense rank of a marked token: marked tokens below it.
__device__ __forceinline__ unsigned mark_rank(const SampleSmem& sm, uint32_t tok) {
  return sm.wordpre[tok >> 5] + (unsigned)__popc(sm.pbits[tok >> 5] & ((1u << (tok & 31u)) - 1u));
}

// gpt2.rs:909-921: for every token of the history (prompt and generated),
// logit /= penalty if it is positive, else logit *= penalty, once per
// occurrence. Per round of token ids (all of them at once while the history
// has at most DMAX entries): the history's tokens are marked in an LDS bitmap,
// the marks ranked densely (prefix popcounts of the words) and counted per
// rank; one thread per marked token applies its occurrences to the logit as
// loaded, and every element reads its result by rank.
template <int NJ>
__device__ __forceinline__ void apply_penalty(float (&v)[NJ], const float* logits, int V, const uint32_t* prompt,
                                              int n_prompt, const uint32_t* ids, int nh, float pen, SampleSmem& sm) {
  const int t = threadIdx.x;
  const int span = nh <= DMAX ? V : DMAX;  // token ids per round: at most DMAX marks
  constexpr int WPT = PBW / ST;            // bitmap words per thread in the scan
  for (int lo = 0; lo < V; lo += span) {
    const uint32_t hi = (uint32_t)min(V, lo + span);
    for (int i = t; i < PBW; i += ST) sm.pbits[i] = 0u;
    for (int i = t; i < DMAX; i += ST) sm.cnt[i] = 0u;
    __syncthreads();
    for (int q = t; q < nh; q += ST) {
      const uint32_t tok = hist_at(prompt, n_prompt, ids, q);
      if (tok >= (uint32_t)lo && tok < hi) atomicOr(&sm.pbits[tok >> 5], 1u << (tok & 31u));
    }
    __syncthreads();
    unsigned pc[WPT], s = 0, marks;
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      pc[k] = (unsigned)__popc(sm.pbits[t * WPT + k]);
      s += pc[k];
    }
    unsigned run = block_excl_scan(s, sm, &marks);
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      sm.wordpre[t * WPT + k] = run;
      run += pc[k];
    }
    __syncthreads();
    for (int q = t; q < nh; q += ST) {
      const uint32_t tok = hist_at(prompt, n_prompt, ids, q);
      if (tok >= (uint32_t)lo && tok < hi) atomicAdd(&sm.cnt[mark_rank(sm, tok)], 1u);
    }
    __syncthreads();
    for (unsigned r = t; r < marks; r += ST) {
      int a = 0, b = PBW - 1;  // the last word with wordpre <= r holds mark r
      while (a < b) {
        const int m = (a + b + 1) >> 1;
        if (sm.wordpre[m] <= r) a = m;
        else b = m - 1;
      }
      uint32_t word = sm.pbits[a];
      for (unsigned z = r - sm.wordpre[a]; z > 0; --z) word &= word - 1u;  // drop the lower marks
      float x = logits[a * 32 + __builtin_ctz(word)];
      for (unsigned z = sm.cnt[r]; z > 0; --z) x = x > 0.0f ? x / pen : x * pen;
      sm.val[r] = x;
    }
    __syncthreads();
    // element j * ST + t is bit t % 32 of word j * ST / 32 + t / 32
    const uint32_t below = (1u << (t & 31)) - 1u;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int wi = j * (ST / 32) + (t >> 5);
      const uint32_t word = sm.pbits[wi];
      if ((word >> (t & 31)) & 1u) v[j] = sm.val[sm.wordpre[wi] + (unsigned)__popc(word & below)];
    }
    __syncthreads();
  }
}

// The token of generation index g by passes over the whole row, on this
// workgroup alone.
template <int NJ>
__device__ __forceinline__ uint32_t sample_whole(const float* __restrict__ logits, int V, const uint32_t* __restrict__ prompt,
                                 int n_prompt, const uint32_t* __restrict__ ids, int g, const SampleParams& sp,
                                 SampleSmem& sm) {
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  // v[j] = element j * ST + t ("row" j), in registers for all passes
  float v[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int i = j * ST + t;
    v[j] = i < V ? logits[i] : -INFINITY;
  }
  if (sp.penalty != 1.0f) apply_penalty<NJ>(v, logits, V, prompt, n_prompt, ids, n_prompt + g, sp.penalty, sm);
  uint32_t pick = 0;
  if (sp.temperature <= 0.0f) {
    // ---- greedy: argmax_f32 (gpt2.rs:858-868), strict '>' from -inf, the
    // first index wins, NaN never wins, -0.0 ties with +0.0 (argmax_key.h) ----
    unsigned long long best = 0ull;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int i = j * ST + t;
      if (i < V) {
        const unsigned long long k = argmax_key(v[j], (uint32_t)i);
        best = k > best ? k : best;
      }
    }
    if (t == 0) sm.key = 0ull;
    __syncthreads();
    if (best) atomicMax(&sm.key, best);
    __syncthreads();
    pick = argmax_key_index(sm.key);
  } else {
#pragma unroll
    for (int j = 0; j < NJ; ++j) v[j] = v[j] / sp.temperature;
    float mx;
    if (sp.top_k > 0 && sp.top_k < V) {
      // ---- top-k (gpt2.rs:924-935): threshold = the k-th largest value ----
      float mn = INFINITY;
      mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (v[j] > -INFINITY) {
          mx = fmaxf(mx, v[j]);
          mn = fminf(mn, v[j]);
        }
      block_minmax(mx, mn, sm);
      // round 1: NB linear bins over [mn, mx]; a monotone map, so equal
      // values share a bin and every value in a higher bin is larger
      const float range = mx - mn;
      const float bs = (range > 0.f && range < INFINITY) ? (float)(NB - 1) / range : 0.f;
      hist_begin<NB>(sm);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (j * ST + t < V) atomicAdd(&sm.hist[lin_bin(v[j], mn, bs)], 1u);
      hist_end<NB>(sm, (unsigned)sp.top_k);
      const unsigned b1 = sm.misc[0];  // k < V elements: always found
      unsigned need = (unsigned)sp.top_k - sm.misc[1];
      uint32_t mm[(NJ + 31) / 32];  // members of bin b1
#pragma unroll
      for (int q = 0; q < (NJ + 31) / 32; ++q) mm[q] = 0u;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (j * ST + t < V && lin_bin(v[j], mn, bs) == b1) mm[j >> 5] |= 1u << (j & 31);
      // rounds 2-4: the order-preserving key of the members, 11 + 11 + 10 bits
      hist_begin<2048>(sm);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((mm[j >> 5] >> (j & 31)) & 1u) atomicAdd(&sm.hist[order_key(v[j]) >> 21], 1u);
      hist_end<2048>(sm, need);
      uint32_t prefix = sm.misc[0] << 21;
      need -= sm.misc[1];
      hist_begin<2048>(sm);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((mm[j >> 5] >> (j & 31)) & 1u) {
          const uint32_t k = order_key(v[j]);
          if ((k >> 21) == (prefix >> 21)) atomicAdd(&sm.hist[(k >> 10) & 2047u], 1u);
        }
      hist_end<2048>(sm, need);
      prefix |= sm.misc[0] << 10;
      need -= sm.misc[1];
      hist_begin<1024>(sm);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((mm[j >> 5] >> (j & 31)) & 1u) {
          const uint32_t k = order_key(v[j]);
          if ((k >> 10) == (prefix >> 10)) atomicAdd(&sm.hist[k & 1023u], 1u);
        }
      hist_end<1024>(sm, need);
      prefix |= sm.misc[0];
      const float thr = from_order_key(prefix);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (v[j] < thr) v[j] = -INFINITY;
    } else {
      mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < NJ; ++j) mx = fmaxf(mx, v[j]);
      mx = block_max(mx, sm);
    }
    // From here v holds e = exp(y - max) of the filtered logits y (0 for the
    // removed ones), proportional to the probabilities p = e / S. Top-p keeps
    // the largest probability, so the maximum of what it leaves is the same,
    // and the distribution sample_from_logits draws from is e / (kept sum):
    // top-p zeroes entries in place.
#pragma unroll
    for (int j = 0; j < NJ; ++j) v[j] = v[j] > -INFINITY ? expf(v[j] - mx) : 0.f;
    float S = seg_total<NJ>(v, sm, w, lane);
    // ---- top-p (gpt2.rs:939-970): keep the largest probabilities, ties in
    // index order, until their running sum reaches p ----
    if (sp.top_p < 1.0f && sp.top_p > 0.0f) {
      // radix descent over the bits of e (non-negative floats order like their
      // bits), 10 + 11 + 10 bits, for the cut-off value with
      // mass(e > cut) < top_p <= mass(e >= cut); masses are summed as
      // integers (p * 2^31 rounded to nearest, mass_of): the same total in
      // any order
      const float ms = 2147483648.0f / S;  // 2^31 / S
      const unsigned target = max(1u, (unsigned)(sp.top_p * 2147483648.0f));
      hist_begin<1024>(sm);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (v[j] > 0.f) atomicAdd(&sm.hist[__float_as_uint(v[j]) >> 21], mass_of(v[j], ms));
      hist_end<1024>(sm, target);
      const uint32_t b1 = sm.misc[0];
      if (b1 != NONE) {  // else the total stays below p: everything is kept
        unsigned above = sm.misc[1];
        hist_begin<2048>(sm);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint32_t k = __float_as_uint(v[j]);
          if (k != 0u && (k >> 21) == b1) atomicAdd(&sm.hist[(k >> 10) & 2047u], mass_of(v[j], ms));
        }
        hist_end<2048>(sm, target - above);
        const uint32_t p21 = (b1 << 11) | sm.misc[0];
        above += sm.misc[1];
        hist_begin<1024>(sm);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint32_t k = __float_as_uint(v[j]);
          if (k != 0u && (k >> 10) == p21) atomicAdd(&sm.hist[k & 1023u], mass_of(v[j], ms));
        }
        hist_end<1024>(sm, target - above);
        const uint32_t cut = (p21 << 10) | sm.misc[0];
        above += sm.misc[1];
        const unsigned qcut = mass_of(__uint_as_float(cut), ms);
        // entries equal to the cut-off all weigh qcut; the first `take` of them
        // in index order are kept, as many as the running sum needs to reach p
        const unsigned take = qcut ? (target - above + qcut - 1) / qcut : 0xffffffffu;
        const unsigned ties = qcut ? sm.misc[2] / qcut : 0xffffffffu;
        if (qcut == 0u || ties <= take) {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            if (__float_as_uint(v[j]) < cut) v[j] = 0.f;
        } else {
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const unsigned long long bal = __ballot(__float_as_uint(v[j]) == cut);
            if (lane == 0) sm.seg[j * SW + w] = (float)__popcll(bal);
          }
          __syncthreads();
          if (w == 0) wave_excl_prefix(sm.seg, sm.segpre, NJ * SW, lane);
          __syncthreads();
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const uint32_t k = __float_as_uint(v[j]);
            const bool tie = k == cut;
            const unsigned long long bal = __ballot(tie);
            bool keep = k > cut;
            if (tie) keep = (unsigned)sm.segpre[j * SW + w] + (unsigned)lanes_before(bal) < take;
            if (!keep) v[j] = 0.f;
          }
        }
        S = seg_total<NJ>(v, sm, w, lane);
      }
    }
    // ---- sample_from_logits (gpt2.rs:973-993): the first index whose
    // running sum of probabilities exceeds the uniform draw, here the first
    // whose running sum of e exceeds draw * S ----
    const float r = (float)(splitmix_at(sp.seed, (uint64_t)sp.draw0 + (uint64_t)g + 1) >> 40) * (1.0f / 16777216.0f);
    const float rs = r * S;
    if (w == 0) {
      // the (row, wave) segment of 64 indices where the running sum first exceeds rs
      const int n = NJ * SW;
      const int per = (n + 63) / 64, b0 = lane * per, e0 = min(n, b0 + per);
      int found = -1;
      for (int i = b0; i < e0 && found < 0; ++i)
        if (rs < sm.segpre[i] + sm.seg[i]) found = i;
      const unsigned long long bal = __ballot(found >= 0);
      const int segi = bal ? __shfl(found, __builtin_ctzll(bal), 64) : -1;
      if (lane == 0) {
        sm.misc[3] = segi < 0 ? NONE : (unsigned)segi;
        sm.fmisc[0] = segi < 0 ? 0.f : sm.segpre[segi];
      }
    }
    __syncthreads();
    const unsigned seg = sm.misc[3];
    if (seg == NONE) {
      pick = (uint32_t)(V - 1);
    } else {
      // inside the segment: 64 consecutive indices, held by wave seg % SW in row seg / SW
      if (w == (int)(seg % SW)) {
        const int row = (int)(seg / SW);
        float p = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (j == row) p = v[j];
        const int i = row * ST + t;
        float incl = p;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const float u = __shfl_up(incl, o, 64);
          if (lane >= o) incl += u;
        }
        const unsigned long long bal = __ballot(i < V && rs < sm.fmisc[0] + incl);
        // the segment's sum (a tree) put rs inside it; should the running sum
        // (another order) stop short by rounding, the segment's last index of
        // non-zero probability is the one the draw falls on
        const unsigned long long nz = __ballot(i < V && p > 0.f);
        const int i0 = row * ST + (int)(seg % SW) * 64;
        if (lane == 0)
          sm.misc[4] = bal ? (unsigned)(i0 + __builtin_ctzll(bal))
                           : nz ? (unsigned)(i0 + 63 - __builtin_clzll(nz)) : (unsigned)(V - 1);
      }
      __syncthreads();
      pick = sm.misc[4];
    }
  }
  return pick;
}

// ---- the same choice over many workgroups and few candidates ----
//
// sample_segments_kernel: workgroup b takes 1024 consecutive logits, applies
// the penalty and the temperature, and leaves the scaled logits y and, per
// segment of 64 consecutive ones, their maximum. sample_pick_kernel, one
// workgroup, then reads the <= 1024 segment records and only the segments that
// matter:
//  - top-k: a segment whose maximum is below k others' holds none of the k
//    largest, so about k segments are read (those that reach a bound just
//    below the k-th largest maximum); of these, values below the bound are
//    dropped. What is left (about k values) is ranked by comparing all pairs, for top-k (fewer than k
//    larger) and for top-p (the mass ranked before it below p, the rule of the
//    histogram rounds above: masses are integers).
//  - no filter: sample_sums_kernel, between the two, adds up every segment's
//    exp(y - maximum of the row); then the segment where the running sum passes
//    the draw.
//  - greedy: the segments' best keys.
// The segments are the (row, wave) segments of the passes above, summed by the
// same tree, and their prefix runs over the same entries, so that every sum and
// with it every pick is the whole row's, bit for bit: with sums in another
// order one draw in a few thousand over a flat row fell on the next token.
// More candidates than fit (many ties), infinities and NaN take the passes
// over the whole row above, in the same launch.
// One workgroup's VALU and LDS atomics bounded the whole-row passes: GPT-2's
// 50257 logits with top-k 50, top-p 0.95 and a penalty took 73 us per token, now
// 4.9 (segments) + 22.7 (pick; 14.9 without top-p), most of the latter the
// latency of its own instruction fetches and of the chain of LDS and memory round
// trips (17.3 with sums over the survivors alone, in another order);
// temperature alone 23.5 us, now 4.8 + 4.9 (sums) + 6.0.
constexpr int SEG = 64, SEGS_MAX = MAX_ROWS * ST / SEG;  // 1024
constexpr int AT = 256, AW = 1024;                       // threads and logits of one segment workgroup
constexpr int CREG = 16;                                 // candidate values per thread: 8192 in 128 segments
constexpr int SURV = 512;                                // values ranked

struct SampleWork {
  float* y;                     // [V] scaled logits
  float* segmax;                // [segments]; NaN where the segment holds one
  float* segsum;                // [segments] no filter: sum of exp(y - maximum of the row)
  unsigned long long* segkey;   // [segments] greedy: best argmax key
};

__host__ __device__ inline size_t align256(size_t x) { return (x + 255) / 256 * 256; }
__host__ __device__ inline SampleWork sample_work(void* mem, int V) {
  char* p = static_cast<char*>(mem);
  const size_t nseg = (size_t)(V + SEG - 1) / SEG;
  SampleWork w;
  w.y = reinterpret_cast<float*>(p);
  p += align256((size_t)V * 4);
  w.segmax = reinterpret_cast<float*>(p);
  p += align256(nseg * 4);
  w.segsum = reinterpret_cast<float*>(p);
  p += align256(nseg * 4);
  w.segkey = reinterpret_cast<unsigned long long*>(p);
  return w;
}

__global__ __launch_bounds__(AT) void sample_segments_kernel(const float* __restrict__ logits, int V,
                                                             const uint32_t* __restrict__ prompt, int n_prompt,
                                                             const uint32_t* __restrict__ ids,
                                                             const int* __restrict__ step_dev, float temperature,
                                                             float penalty, SampleWork wk) {
  __shared__ unsigned cnt[AW];
  constexpr int R = AW / AT;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int base = blockIdx.x * AW, first = base + wave * (R * 64);
  float x[R];
#pragma unroll
  for (int r = 0; r < R; ++r) x[r] = logits[min(first + r * 64 + lane, V - 1)];
  if (penalty != 1.0f) {
    // gpt2.rs:909-921, once per occurrence of a token in the history
    const int nh = n_prompt + *step_dev - 1;
#pragma unroll
    for (int i = 0; i < R; ++i) cnt[t + i * AT] = 0u;
    __syncthreads();
    for (int q = t; q < nh; q += AT) {
      const uint32_t off = hist_at(prompt, n_prompt, ids, q) - (uint32_t)base;
      if (off < (uint32_t)AW) atomicAdd(&cnt[off], 1u);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
      for (unsigned z = cnt[wave * (R * 64) + r * 64 + lane]; z > 0; --z)
        x[r] = x[r] > 0.0f ? x[r] / penalty : x[r] * penalty;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = first + r * 64 + lane, seg = i / SEG;
    if (first + r * 64 >= V) break;  // wave-uniform
    if (temperature <= 0.0f) {
      unsigned long long k = i < V ? argmax_key(x[r], (uint32_t)i) : 0ull;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long u = __shfl_xor(k, o, 64);
        k = u > k ? u : k;
      }
      if (lane == 0) wk.segkey[seg] = k;
      continue;
    }
    const float y = i < V ? x[r] / temperature : -INFINITY;
    if (i < V) wk.y[i] = y;
    const float m = wave_max_s(y);
    const bool nan = __any(y != y);
    if (lane == 0) wk.segmax[seg] = nan ? NAN : m;
  }
}

// segsum of the 16 segments of a workgroup, each added up as seg_sums does.
__global__ __launch_bounds__(AT) void sample_sums_kernel(int V, SampleWork wk) {
  __shared__ float red[AT / 64];
  constexpr int R = AW / AT;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nseg = (V + SEG - 1) / SEG;
  const int first = blockIdx.x * AW + wave * (R * 64);
  float y[R], m = -INFINITY;
#pragma unroll
  for (int r = 0; r < R; ++r) y[r] = wk.y[min(first + r * 64 + lane, V - 1)];
#pragma unroll
  for (int r = 0; r < SEGS_MAX / AT; ++r) m = fmaxf(m, wk.segmax[min(t + r * AT, nseg - 1)]);
  m = wave_max_s(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < AT / 64; ++i) m = fmaxf(m, red[i]);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = first + r * 64 + lane;
    if (first + r * 64 >= V) break;  // wave-uniform
    float e = i < V && y[r] > -INFINITY ? expf(y[r] - m) : 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
    if (lane == 0) wk.segsum[i / SEG] = e;
  }
}

struct PickSmem {
  float segmax[SEGS_MAX];
  float seg[SEGS_MAX];     // sums per segment and
  float segpre[SEGS_MAX];  // their exclusive prefix
  uint16_t cand[SEGS_MAX];
  float val[SURV];         // survivors: scaled logits, then exp(y - maximum)
  unsigned mass[SURV];
  float red[2 * SW];
  unsigned wtot[SW];
  float fmisc[2];
  unsigned misc[2];
};

// Exclusive prefix over the block in thread order (as block_excl_scan).
__device__ __forceinline__ unsigned pick_scan(unsigned x, PickSmem& sm, unsigned* total) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned incl = x;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  __syncthreads();
  if (lane == 63) sm.wtot[w] = incl;
  __syncthreads();
  unsigned base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SW; ++i) {
    if (i == w) base = tot;
    tot += sm.wtot[i];
  }
  *total = tot;
  return base + incl - x;
}

// The first of n (<= 1024) segments whose running sum exceeds r * (the sum of
// all), r a uniform draw; NONE when none does. Every thread gets it (and that
// segment's exclusive prefix in *before, the threshold in *rs).
__device__ __forceinline__ uint32_t pick_entry(PickSmem& sm, int n, float r, float* before, float* rs) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (w == 0) {
    const float S = wave_excl_prefix(sm.seg, sm.segpre, n, lane);
    const float lim = r * S;
    const int per = (n + 63) / 64, b0 = lane * per, e0 = min(n, b0 + per);
    int found = -1;
    for (int i = b0; i < e0 && found < 0; ++i)
      if (lim < sm.segpre[i] + sm.seg[i]) found = i;
    const unsigned long long bal = __ballot(found >= 0);
    const int f = bal ? __shfl(found, __builtin_ctzll(bal), 64) : -1;
    if (lane == 0) {
      sm.misc[0] = f < 0 ? NONE : (unsigned)f;
      sm.fmisc[0] = f < 0 ? 0.f : sm.segpre[f];
      sm.fmisc[1] = lim;
    }
  }
  __syncthreads();
  *before = sm.fmisc[0];
  *rs = sm.fmisc[1];
  return sm.misc[0];
}

// One wave, its lanes holding segment seg's p = exp(y - maximum) (0: removed),
// before the running sum up to it: the index where it passes rs. Should the
// running sum stop short of the segment's (a tree) by rounding, its last index
// of non-zero probability.
__device__ __forceinline__ uint32_t pick_in_segment(float p, uint32_t seg, float before, float rs, int V, int lane) {
  float incl = p;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  const unsigned long long bal = __ballot((int)seg * SEG + lane < V && rs < before + incl);
  const unsigned long long nz = __ballot(p > 0.f);
  return bal ? seg * SEG + (uint32_t)__builtin_ctzll(bal)
             : nz ? seg * SEG + 63u - (uint32_t)__builtin_clzll(nz) : (uint32_t)(V - 1);
}

// The pick from the segment records; false when the whole row is needed. NJ:
// registers per thread of sample_whole's row, whose NJ * SW segments the sums
// run over.
template <int NJ>
__device__ __forceinline__ bool pick_from_segments(const SampleWork& wk, int V, int g, const SampleParams& sp, PickSmem& sm,
                                   uint32_t* pick) {
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  constexpr int NS = NJ * SW;  // >= nseg; the segments past the row are empty
  const int nseg = (V + SEG - 1) / SEG;
  const bool top_k = sp.top_k > 0 && sp.top_k < V;
  // segments 2t and 2t + 1 of this thread
  float m2[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = min(2 * t + q, nseg - 1);
    m2[q] = wk.segmax[i];
    float s = top_k ? 0.f : wk.segsum[i];
    if (2 * t + q >= nseg) {
      m2[q] = -INFINITY;
      s = 0.f;
    }
    sm.segmax[2 * t + q] = m2[q];
    sm.seg[2 * t + q] = s;
  }
  float mx = wave_max_s(fmaxf(m2[0], m2[1]));
  const bool bad = __any(m2[0] != m2[0] || m2[1] != m2[1]);
  if (lane == 0) {
    sm.red[w] = mx;
    sm.red[SW + w] = bad ? 1.f : 0.f;
  }
  __syncthreads();
  float any_bad = 0.f;
#pragma unroll
  for (int i = 0; i < SW; ++i) {
    mx = fmaxf(mx, sm.red[i]);
    any_bad += sm.red[SW + i];
  }
  if (any_bad != 0.f || !(fabsf(mx) < INFINITY)) return false;
  const float r =
      (float)(splitmix_at(sp.seed, (uint64_t)sp.draw0 + (uint64_t)g + 1) >> 40) * (1.0f / 16777216.0f);
  float before, rs;
  if (!top_k) {
    // ---- temperature only: the segment, then the index inside it ----
    const uint32_t seg = pick_entry(sm, NS, r, &before, &rs);
    if (seg == NONE) {
      *pick = (uint32_t)(V - 1);
      return true;
    }
    const int i = (int)seg * SEG + lane;
    const float y = i < V ? wk.y[i] : -INFINITY;
    *pick = pick_in_segment(y > -INFINITY ? expf(y - mx) : 0.f, seg, before, rs, V, lane);
    return true;
  }
  // ---- top-k: a bound that at least k segments' maxima reach (the top 16
  // bits of the k-th largest maximum's order key, bit by bit on one wave: all
  // pairs of maxima took 10 us), and the segments that reach it ----
  const int k = sp.top_k;
  if (w == 0) {
    uint32_t key[SEGS_MAX / 64];
#pragma unroll
    for (int j = 0; j < SEGS_MAX / 64; ++j) key[j] = order_key(sm.segmax[64 * j + lane]) >> 16;
    uint32_t bound = 0;
#pragma unroll 1
    for (int bit = 15; bit >= 0; --bit) {
      const uint32_t next = bound | 1u << bit;
      int n = 0;
#pragma unroll
      for (int j = 0; j < SEGS_MAX / 64; ++j) n += __popcll(__ballot(key[j] >= next));
      if (n >= k) bound = next;
    }
    if (lane == 0) sm.misc[0] = bound;
  }
  __syncthreads();
  const uint32_t bound = sm.misc[0];
  float low = from_order_key(bound << 16);
  if (!(low > -INFINITY)) low = -INFINITY;  // (fewer than k finite maxima: they bound nothing)
  unsigned nc;
  const bool c0 = 2 * t < nseg && order_key(m2[0]) >> 16 >= bound;
  const bool c1 = 2 * t + 1 < nseg && order_key(m2[1]) >> 16 >= bound;
  unsigned at = pick_scan((c0 ? 1u : 0u) + (c1 ? 1u : 0u), sm, &nc);
  if (c0) sm.cand[at++] = (uint16_t)(2 * t);
  if (c1) sm.cand[at] = (uint16_t)(2 * t + 1);
  __syncthreads();
  if (nc > (unsigned)(CREG * SW)) return false;
  // candidate c = CREG * wave + j: consecutive per wave, so that survivors
  // gather in index order, lane l holding index l of the segment
  float v[CREG];
  unsigned mine = 0;
#pragma unroll
  for (int j = 0; j < CREG; ++j) {
    const unsigned c = CREG * w + j;
    v[j] = -INFINITY;
    if (c < nc) {
      const int i = (int)sm.cand[c] * SEG + lane;
      if (i < V) v[j] = wk.y[i];
    }
  }
#pragma unroll
  for (int j = 0; j < CREG; ++j) mine += (unsigned)__popcll(__ballot(v[j] >= low && v[j] > -INFINITY));
  __syncthreads();
  if (lane == 0) sm.wtot[w] = mine;
  __syncthreads();
  unsigned pos = 0, ns = 0;
#pragma unroll
  for (int i = 0; i < SW; ++i) {
    if (i == w) pos = ns;
    ns += sm.wtot[i];
  }
  if (ns > (unsigned)SURV) return false;
  int at_val[CREG];  // this lane's survivor of candidate j, or -1
#pragma unroll
  for (int j = 0; j < CREG; ++j) {
    const unsigned long long bal = __ballot(v[j] >= low && v[j] > -INFINITY);
    at_val[j] = (bal >> lane) & 1ull ? (int)pos + lanes_before(bal) : -1;
    if (at_val[j] >= 0) sm.val[at_val[j]] = v[j];
    pos += (unsigned)__popcll(bal);
  }
  __syncthreads();
  // top-k over the survivors: all values with fewer than k larger ones
  const bool have = (unsigned)t < ns;
  const float yv = have ? sm.val[t] : -INFINITY;
  int larger = 0;
#pragma unroll 8
  for (unsigned i = 0; i < ns; ++i) larger += sm.val[i] > yv;
  float e = have && larger < k ? expf(yv - mx) : 0.f;
  // segment sums of the e in sm.val, by seg_sums' tree
  static_assert(CREG == 16, "the transposing butterfly's chunk");
  auto sums = [&]() {
    __syncthreads();  // every thread is done with sm.val and sm.seg
    if (have) sm.val[t] = e;
    __syncthreads();
    float a[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = at_val[j] >= 0 ? sm.val[at_val[j]] : 0.f;
    tr_stage<16, 32>(a, lane);
    tr_stage<8, 16>(a, lane);
    tr_stage<4, 8>(a, lane);
    tr_stage<2, 4>(a, lane);
    a[0] += __shfl_xor(a[0], 2, 64);
    a[0] += __shfl_xor(a[0], 1, 64);
    const unsigned c = CREG * w + (lane >> 2);
    if ((lane & 3) == 0 && c < nc) sm.seg[sm.cand[c]] = a[0];
    __syncthreads();
  };
  sums();
  if (sp.top_p < 1.0f && sp.top_p > 0.0f) {
    if (w == 0) {
      const float S = wave_excl_prefix(sm.seg, sm.segpre, NS, lane);
      if (lane == 0) sm.fmisc[0] = S;
    }
    __syncthreads();
    const float ms = 2147483648.0f / sm.fmisc[0];
    const unsigned target = max(1u, (unsigned)(sp.top_p * 2147483648.0f));
    if (have) sm.mass[t] = mass_of(e, ms);
    __syncthreads();
    unsigned before_mass = 0;
#pragma unroll 8
    for (unsigned i = 0; i < ns; ++i) {
      const float o = sm.val[i];
      if (o > e || (o == e && i < (unsigned)t)) before_mass += sm.mass[i];
    }
    if (before_mass >= target) e = 0.f;
    sums();
  }
  const uint32_t seg = pick_entry(sm, NS, r, &before, &rs);
  if (seg == NONE) {
    *pick = (uint32_t)(V - 1);
    return true;
  }
  // (the wave that holds the segment; each is a candidate once)
#pragma unroll
  for (int j = 0; j < CREG; ++j)
    if (CREG * w + j < (int)nc && sm.cand[CREG * w + j] == seg) {  // wave-uniform
      const uint32_t i = pick_in_segment(at_val[j] >= 0 ? sm.val[at_val[j]] : 0.f, seg, before, rs, V, lane);
      if (lane == 0) sm.misc[1] = i;
    }
  __syncthreads();
  *pick = sm.misc[1];
  return true;
}

template <int NJ>
__global__ __launch_bounds__(ST) void sample_kernel(const float* __restrict__ logits, int V,
                                                    const uint32_t* __restrict__ prompt, int n_prompt,
                                                    uint32_t* __restrict__ ids, const int* __restrict__ step_dev,
                                                    SampleParams sp, uint32_t* __restrict__ token) {
  __shared__ SampleSmem sm;
  const int g = *step_dev - 1;  // generation index of the token being chosen
  const uint32_t pick = sample_whole<NJ>(logits, V, prompt, n_prompt, ids, g, sp, sm);
  if (threadIdx.x == 0) {
    token[0] = pick;
    ids[g] = pick;
  }
}

template <int NJ>
__global__ __launch_bounds__(ST) void sample_pick_kernel(const float* __restrict__ logits, int V,
                                                         const uint32_t* __restrict__ prompt, int n_prompt,
                                                         uint32_t* __restrict__ ids,
                                                         const int* __restrict__ step_dev, SampleParams sp,
                                                         uint32_t* __restrict__ token, SampleWork wk) {
  __shared__ __attribute__((aligned(16))) union {
    SampleSmem whole;
    PickSmem part;
  } sm;
  const int t = threadIdx.x, lane = t & 63;
  const int g = *step_dev - 1;  // generation index of the token being chosen
  uint32_t pick = 0;
  if (sp.temperature <= 0.0f) {
    const int nseg = (V + SEG - 1) / SEG;
    unsigned long long k = 0ull;
    for (int i = t; i < nseg; i += ST) k = wk.segkey[i] > k ? wk.segkey[i] : k;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const unsigned long long u = __shfl_xor(k, o, 64);
      k = u > k ? u : k;
    }
    if (t == 0) sm.whole.key = 0ull;
    __syncthreads();
    if (lane == 0) atomicMax(&sm.whole.key, k);
    __syncthreads();
    pick = argmax_key_index(sm.whole.key);
  } else if (!pick_from_segments<NJ>(wk, V, g, sp, sm.part, &pick)) {
    __syncthreads();
    pick = sample_whole<NJ>(logits, V, prompt, n_prompt, ids, g, sp, sm.whole);
  }
  if (t == 0) {
    token[0] = pick;
    ids[g] = pick;
  }
}

}  // namespace

size_t sample_work_bytes(int V) {
  const size_t nseg = (size_t)(V + SEG - 1) / SEG;
  return align256((size_t)V * 4) + 2 * align256(nseg * 4) + align256(nseg * 8);
}

bool launch_sample(hipStream_t s, const float* logits, int V, const uint32_t* prompt, int n_prompt, uint32_t* ids,
                   const int* step_dev, const SampleParams& sp, uint32_t* token, void* work) {
  if (V <= 0 || V > MAX_ROWS * ST) return false;
  // Segments for rows that one workgroup takes long over, unless top-p alone
  // filters (its kept set is most of a flat row) or top-k keeps more than the ranking
  // is made for.
  const bool top_k = sp.top_k > 0 && sp.top_k < V, top_p = sp.top_p < 1.0f && sp.top_p > 0.0f;
  const bool segments =
      work != nullptr && V > 4 * ST && (sp.temperature <= 0.0f || (top_k ? sp.top_k <= SURV / 4 : !top_p));
  const SampleWork wk = sample_work(work, V);
  if (segments)
    sample_segments_kernel<<<(V + AW - 1) / AW, AT, 0, s>>>(logits, V, prompt, n_prompt, ids, step_dev,
                                                            sp.temperature, sp.penalty, wk);
  if (segments && !top_k && sp.temperature > 0.0f)
    sample_sums_kernel<<<(V + AW - 1) / AW, AT, 0, s>>>(V, wk);
#define RTG_SAMPLE(NJ)                                                                                         \
  do {                                                                                                         \
    if (segments)                                                                                              \
      sample_pick_kernel<NJ><<<1, ST, 0, s>>>(logits, V, prompt, n_prompt, ids, step_dev, sp, token, wk);      \
    else                                                                                                       \
      sample_kernel<NJ><<<1, ST, 0, s>>>(logits, V, prompt, n_prompt, ids, step_dev, sp, token);               \
  } while (0)
  if (V <= 1 * ST) RTG_SAMPLE(1);
  else if (V <= 4 * ST) RTG_SAMPLE(4);
  else if (V <= 16 * ST) RTG_SAMPLE(16);
  else if (V <= 64 * ST) RTG_SAMPLE(64);
  else if (V <= 100 * ST) RTG_SAMPLE(100);  // GPT-2's 50257 tokens
  else RTG_SAMPLE(128);
#undef RTG_SAMPLE
  return true;
}

}  // namespace rtg
