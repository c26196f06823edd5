// How the fp32 GEMMs are cut into workgroups: host code without HIP includes.
#pragma once

#include <algorithm>
#include <cstdint>
#include <iterator>

#include "fastdiv.hpp"

namespace lmp_hip {

// A grid holds fewer than 2^32 threads per dimension: a dispatch counts them in
// 32 bits, and a longer one-shot launch comes out as what is left modulo 2^32
// (2^33 + 64 threads as a single wave).
constexpr uint64_t kMaxGridThreads = 0xffffffffull;

// `blocks` workgroups over two dimensions of a grid, y past 1 only where x alone
// would have too many threads; block y * x_extent + x may lie past the last one.
struct Grid2 {
  uint32_t x = 1, y = 1;
};
inline Grid2 grid_2d(uint64_t blocks, int threads) {
  const uint64_t most = kMaxGridThreads / uint64_t(threads);
  const uint64_t y = (blocks + most - 1) / most;
  return {uint32_t((blocks + y - 1) / y), uint32_t(y)};
}

// ------------------------------------------------------- products of up to 32 rows

// K split over workgroups, `per_wg` values each; a workgroup's `waves` waves take
// consecutive parts of its range.
struct KSplit {
  int splits = 1, per_wg = 0;
};

// One past the last k of a wave that takes `part` values from `kb` on: at most
// k, and no more than kb for a wave past the end (kb + part may not fit an int).
LMP_HD int k_range_end(int kb, int part, int k) {
  const int left = k - kb;
  return kb + (part < left ? part : left);
}

constexpr int kRowsWaves = 4;

// A workgroup for every 32 of n columns fits a grid.
inline bool rows_fit(int64_t n) {
  return uint64_t(n + 31) / 32 <= kMaxGridThreads / (64 * kRowsWaves);
}

// Rows kernel (B transposed, one workgroup per 32 columns).  A CU holds one
// workgroup, so the split count is the one whose rounds of workgroups take the
// fewest tile steps: a step of the whole chip (4 MiB of B) is about 1 us, as
// are a round's start and end, and folding partials costs about 4.
inline KSplit rows_split(int64_t cus, int64_t n, int64_t k) {
  constexpr int64_t kGrain = 32 * kRowsWaves;
  const int64_t blocks = (n + 31) / 32;
  const int64_t k_tiles = (k + kGrain - 1) / kGrain;  // a wave's tiles, unsplit
  int64_t per = k_tiles, best = INT64_MAX;
  const int64_t max_splits =
      std::max<int64_t>(1, std::min<int64_t>(k_tiles / 2, 2 * cus / blocks));
  for (int64_t s = 1; s <= max_splits; ++s) {
    const int64_t steps = (k_tiles + s - 1) / s;
    const int64_t rounds = (blocks * s + cus - 1) / cus;
    const int64_t cost = rounds * (steps + 1) + (s > 1 ? 4 : 0);
    if (cost < best) {
      best = cost;
      per = steps;
    }
  }
  return {int((k_tiles + per - 1) / per), int(per * kGrain)};
}

constexpr int kDirectWaves = 4;

// Register-direct kernel: `splits` workgroups (0: enough for the CUs) of 64 k or
// more per wave for each of `blocks` column blocks.
inline KSplit direct_split(int64_t cus, int64_t blocks, int64_t k, int64_t splits) {
  constexpr int64_t kGrain = 8 * kDirectWaves;
  const int64_t most = std::max<int64_t>(1, k / (64 * kDirectWaves));
  if (splits <= 0) splits = (cus + blocks - 1) / blocks;
  splits = std::max<int64_t>(1, std::min(splits, most));
  const int64_t per = ((k + splits - 1) / splits + kGrain - 1) / kGrain * kGrain;
  return {int((k + per - 1) / per), int(per)};
}

// ---------------------------------------------- products on the bf16 matrix cores

constexpr int kBf3K = 16;  // k values per step

struct Bf3Plan {
  int cfg = -1;  // index into kBf3Tiles; -1: no launch fits a grid
  int splits = 1;
};

// Time of one 16-wide k step of a workgroup, in us: `alone` on its CU, and
// `shared` per workgroup where several take turns (fitted to a sweep of 66
// products over every tile and split, random operands, on one MI355X: the plan
// takes 0.4% more than the best of the sweep, 8% at worst).  A larger tile moves
// and splits each value fewer times: 4096^3 takes 565-640, 650-680, 710-780,
// 870 and about 980 us on the five, 512 x 1000 x 4096 (K split) 44, 37, 34, 37,
// 38 and 256 x 1024 x 1024 25, 19, 16, 15.5, 14.
// APART: the leading products of a value accumulate apart from the small ones,
// one rounding of the sum a step (six without, which the largest tile's
// accumulators leave no registers for).
struct Bf3Tile {
  int bm, bn, threads;
  bool apart;
  float alone, shared;
};
constexpr Bf3Tile kBf3Tiles[] = {{256, 256, 512, false, 1.78f, 2.4f},
                                 {256, 128, 512, true, 1.07f, 1.45f},
                                 {128, 128, 512, true, 0.61f, 0.75f},
                                 {64, 128, 256, true, 0.475f, 0.441f},
                                 {64, 64, 256, true, 0.26f, 0.252f}};

inline int64_t bf3_tiles(const Bf3Tile& t, int64_t m, int64_t n) {
  return ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
}

// Tiles and split of K with the least modelled time: workgroups go round the
// CUs, each takes 4.5 us besides its steps (first loads, C), and a split costs
// a second launch (2 us) and a round trip of the partials (5 TB/s).  The
// partials stay within `scratch` bytes, the fixed workspace, whichever entry
// point is called, so that all of them give the same bits; a split keeps at
// least 64 k.  Launches that a grid cannot hold are left out, and the tile with
// one accumulator where it would not give every CU one: there the fp32 kernels
// split K, and their shorter chains round less than its long one (2048^3: 5.7e-7
// from float64 in two splits, 7.0e-7 here unsplit, 2.7e-7 with sums apart).
inline Bf3Plan bf3_plan(int64_t cus, int64_t scratch, int64_t m, int64_t n, int64_t k) {
  const int64_t steps = (k + kBf3K - 1) / kBf3K, mn = m * n;
  const int64_t most =
      std::min<int64_t>(std::max<int64_t>(1, steps / 4),
                        scratch / int64_t(sizeof(float)) /
                            (mn + n + 8));  // room for column sums, asked for or not
  Bf3Plan plan;
  float best = 0.0f;
  for (int c = 0; c < int(std::size(kBf3Tiles)); ++c) {
    const Bf3Tile& t = kBf3Tiles[c];
    const int64_t tiles = bf3_tiles(t, m, n);
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64}) {
      if (s > 1 && (s > most || !t.apart)) break;
      if (!t.apart && tiles < cus) break;
      if (uint64_t(tiles) * uint64_t(s) > kMaxGridThreads / uint64_t(t.threads)) break;
      const float load = float((tiles * s + cus - 1) / cus);
      const float per_step = std::max(t.alone, load * t.shared);
      float us = 4.5f + float((steps + s - 1) / s) * per_step;
      if (s > 1) us += 2.0f + float(s + 1) * float(mn) * (4.0f / 5e6f);
      if (plan.cfg < 0 || us < best) {
        best = us;
        plan.cfg = c;
        plan.splits = s;
      }
      if (tiles * s > 8 * cus) break;  // more splits only add partials
    }
  }
  return plan;
}

// Whether two planned products of `a` and `b` workgroups fit one grid.
inline bool bf3_pair_fits(uint64_t a, uint64_t b, int threads) {
  return a + b <= kMaxGridThreads / uint64_t(threads);
}

}  // namespace lmp_hip
