// Host-only checks of how the fp32 GEMMs are cut into workgroups.  Built and run
// by tests/test_gemm_plan.py with g++; no GPU involved.
#include <cstdio>

#include "gemm_plan.hpp"

using namespace lmp_hip;

#define CHECK(c)                                                  \
  do {                                                            \
    if (!(c)) {                                                   \
      std::printf("FAIL %s:%d %s\n", __FILE__, __LINE__, #c);     \
      return 1;                                                   \
    }                                                             \
  } while (0)

constexpr int64_t kTop = (int64_t(1) << 31) - 4097;  // the largest extent a GEMM takes
constexpr int64_t kScratch = int64_t(32) << 20;

// Every launch of the bf16 path has fewer than 2^32 threads, at any extents.
int bf3_grids() {
  const int64_t ms[] = {33, 512, 4096, int64_t(1) << 24, (int64_t(1) << 30) - 64, int64_t(1) << 30,
                        (int64_t(1) << 30) + 64, kTop - 255, kTop};
  const int64_t ns[] = {1, 64, 65, 128, 129, 4096};
  for (int64_t m : ms)
    for (int64_t n : ns)
      for (int64_t k : {int64_t(33), int64_t(48), int64_t(1000), int64_t(1) << 20})
        for (int flip = 0; flip < 2; ++flip) {
          const int64_t a = flip ? n : m, b = flip ? m : n;
          const Bf3Plan p = bf3_plan(256, kScratch, a, b, k);
          if (p.cfg < 0) {  // only where no tile fits a grid
            for (const Bf3Tile& t : kBf3Tiles)
              CHECK(bf3_tiles(t, a, b) * t.threads > int64_t(kMaxGridThreads));
            continue;
          }
          const Bf3Tile& t = kBf3Tiles[p.cfg];
          CHECK(bf3_tiles(t, a, b) * p.splits * t.threads <= int64_t(kMaxGridThreads));
        }
  // What memory can hold is served: 2^30 + 64 rows of one column (33 values of k
  // each), and the longest extent with up to a tile of the other.
  CHECK(bf3_plan(256, kScratch, (int64_t(1) << 30) + 64, 1, 33).cfg >= 0);
  CHECK(bf3_plan(256, kScratch, kTop, 64, 33).cfg >= 0);
  CHECK(bf3_plan(256, kScratch, 64, kTop, 33).cfg >= 0);
  return 0;
}

// The tile with one accumulator: whole K, and a tile for every CU.
int bf3_sums_apart() {
  for (int64_t m : {64, 512, 1000, 2048, 4000, 4096, 8192, 20000})
    for (int64_t n : {64, 1000, 2048, 4096, 8192})
      for (int64_t k : {33, 64, 512, 4096, 100000}) {
        const Bf3Plan p = bf3_plan(256, kScratch, m, n, k);
        CHECK(p.cfg >= 0);
        const Bf3Tile& t = kBf3Tiles[p.cfg];
        CHECK(t.apart || (p.splits == 1 && bf3_tiles(t, m, n) >= 256));
      }
  CHECK(!kBf3Tiles[bf3_plan(256, kScratch, 4096, 4096, 4096).cfg].apart);
  CHECK(kBf3Tiles[bf3_plan(256, kScratch, 2048, 2048, 2048).cfg].apart);
  return 0;
}

// Two products share a launch only where their workgroups together fit a grid.
int bf3_pairs() {
  CHECK(bf3_pair_fits(1, 1, 512));
  const uint64_t most = kMaxGridThreads / 256;
  CHECK(bf3_pair_fits(most - 5, 5, 256) && !bf3_pair_fits(most - 5, 6, 256));
  return 0;
}

// The waves of the kernels for up to 32 rows cover K once: consecutive ranges,
// none past the end (the last workgroup's may start close to 2^31).
int covers(const KSplit& s, int waves, int64_t k) {
  CHECK(s.splits >= 1 && s.per_wg > 0 && s.per_wg % waves == 0);
  const int part = s.per_wg / waves;
  int64_t at = 0;
  for (int y = 0; y < s.splits; ++y)
    for (int w = 0; w < waves; ++w) {
      const int64_t kb64 = int64_t(y) * s.per_wg + int64_t(w) * part;
      CHECK(kb64 < (int64_t(1) << 31));
      const int kb = int(kb64), ke = k_range_end(kb, part, int(k));
      if (ke <= kb) continue;  // a wave past the end
      CHECK(kb == at);
      at = ke;
    }
  CHECK(at == k);
  return 0;
}

int thin_ranges() {
  for (int64_t k : {int64_t(4), int64_t(128), int64_t(388), int64_t(8200), int64_t(1) << 30, kTop - 32768,
                    kTop - 30000, kTop - 4096, kTop - 4, kTop})
    for (int64_t n : {int64_t(1), int64_t(32), int64_t(33), int64_t(100), int64_t(1000), int64_t(4098),
                      int64_t(8192), int64_t(8224), int64_t(100000)})
      for (int64_t cus : {int64_t(256), int64_t(304), int64_t(64)}) {
        if (covers(rows_split(cus, n, k), kRowsWaves, k)) return 1;
        if (covers(direct_split(cus, (n + 127) / 128, k, 0), kDirectWaves, k)) return 1;
      }
  return 0;
}

// grid_2d: every block, fewer than 2^32 threads a dimension, less than one row over.
int grids() {
  for (uint64_t blocks : {uint64_t(1), uint64_t(1000), (uint64_t(1) << 24) - 1, uint64_t(1) << 24,
                          (uint64_t(1) << 24) + 1, uint64_t(1) << 29, uint64_t(0x7fffffff)}) {
    const Grid2 g = grid_2d(blocks, 256);
    CHECK(uint64_t(g.x) * 256 <= kMaxGridThreads && g.y <= 65535);
    CHECK(uint64_t(g.x) * g.y >= blocks && uint64_t(g.x) * g.y - blocks < g.x);
    CHECK(g.y == 1 || blocks * 256 > kMaxGridThreads);
  }
  CHECK(rows_fit(8192) && rows_fit((int64_t(1) << 29) - 32) && !rows_fit(int64_t(1) << 29));
  return 0;
}

int main() {
  if (bf3_grids() || bf3_sums_apart() || bf3_pairs() || thin_ranges() || grids()) return 1;
  std::printf("gemm plans ok\n");
  return 0;
}
