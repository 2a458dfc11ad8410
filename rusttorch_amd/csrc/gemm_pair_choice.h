// Which tile and k split a prefill GEMM on f16 pairs runs (gemm_pair.hip); host
// code without HIP, so that a test can check what the dispatch reaches.
#pragma once
#include <stddef.h>

#include <algorithm>

namespace rtg {

// The tiles, and their times per k-tile of 32 with two planes (us): alone on a
// CU, and per workgroup where a CU has several to run. Fitted to a sweep of
// every tile and split over the GPT-2 widths' GEMMs at 48 to 16368 rows: the
// choice below is within 2% of each shape's fastest in the mean, 8-28% at
// worst (333 x 3072 x 768: 17.3 against 13.5 us).
// What each is for (us, f32 weights, M x N x K, tile against the next best):
//   256 x 256: 16368 x 5120 x 1280: 567 (378 TFLOP/s) against 642
//   128 x 128, two per CU: 16368 x 1280 x 5120: 630 against 702
//   128 x 128 on 8 waves: 701 x 4096 x 1024: 28.2 against 31.9
//   64 x 128: 3000 x 1280 x 1280: 40.0, 701 x 3072 x 1024: 27.6 against 30.0
//   64 x 64: 333 x 3072 x 768: 13.5 against 17.3
//   32 x 64: 77 x 5120 x 1280: 14.3 against 16.4
// (f32-MFMA kernels before: 16368 x 5120 x 1280 1704-1926 us, 701 x 4096 x
// 1024 74, 77 x 5120 x 1280 49.)
struct PairTile {
  int bm, bn;
  float alone, shared;
};
constexpr PairTile kPairTiles[] = {
    {256, 256, 2.30f, 2.60f},  // 0: 8 waves of 128 x 64, 2 stages
    {128, 128, 1.00f, 0.72f},  // 1: 4 waves of 64 x 64, 2 stages, two workgroups per CU
    {128, 128, 0.69f, 0.78f},  // 2: 8 waves of 64 x 32, 3 stages
    {64, 128, 0.40f, 0.44f},   // 3: 4 waves of 64 x 32, 3 stages
    {64, 64, 0.28f, 0.27f},    // 4: 8 waves of 32 x 32 (KW = 2), 4 stages
    {32, 64, 0.20f, 0.20f},    // 5: 4 waves of 32 x 32 (KW = 2), 6 stages
};
constexpr int kSplitMaxRows = 2048;                   // more rows fill the GPU without a split
constexpr size_t kSplitMaxFloats = (size_t)16 << 20;  // and no larger workspace than this

struct PairChoice {
  int tile, ks;
};

// Tile and k split with the least estimated time: the k-tiles of a workgroup
// times the time of one with the workgroups its CU holds, over 256 CUs, plus
// the split's reduction (a launch, and its partials' way through memory).
// Depends on M through its blocks of 32 rows only.
inline PairChoice pair_choose(int M, int N, int K, int planes, size_t ws_floats) {
  const int mr = (M + 31) / 32 * 32, nk = K / 32;
  PairChoice best{5, 1};
  float least = 1e30f;
  for (int c = 0; c < (int)(sizeof(kPairTiles) / sizeof(kPairTiles[0])); ++c) {
    const PairTile& t = kPairTiles[c];
    const long tiles = (long)((mr + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    for (int ks = 1; ks <= 10; ++ks) {
      const size_t floats = (size_t)ks * mr * N;
      if (nk % ks != 0) continue;
      if (ks > 1 && (mr > kSplitMaxRows || floats > kSplitMaxFloats || (size_t)ks * M * N > ws_floats)) break;
      const long per_cu = (tiles * ks + 255) / 256;
      const float step = (planes == 2 ? 1.f : 0.7f) * std::max(t.alone, per_cu * t.shared);
      const float us = nk / ks * step + (ks > 1 ? 2.f + floats * 4 / 3.6e6f : 0.f);
      if (us < least) {
        least = us;
        best = {c, ks};
      }
    }
  }
  return best;
}

}  // namespace rtg
