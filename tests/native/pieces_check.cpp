// Checks of the pieces of crowded tiles (csrc/pm_pieces.h) for random and extreme tile fillings: what the scan
// lists and reserves stays within its arrays, and tiles' blocks and pieces take every entry exactly once.
//   pieces_check SEED      exits 0 when all hold
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "pm_pieces.h"

using namespace pm;

#define CHECK(cond)                                                   \
  do {                                                                \
    if (!(cond)) {                                                    \
      std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond);   \
      return 1;                                                       \
    }                                                                 \
  } while (0)

// counts: entries of every key (own keys, then halo keys); the lists as the scan makes them, in any order
static int check(long np, long ntiles, bool halo, const std::vector<uint32_t>& counts, std::mt19937& rng) {
  const PieceSizes s = piece_sizes(np, ntiles, halo);
  CHECK(s.per >= kRefPiece && s.dense >= 2 * s.per && s.parts <= s.max && s.parts <= 2 * kRefPieces);
  std::vector<size_t> order(counts.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::shuffle(order.begin(), order.end(), rng);
  uint32_t listed = 0, taken = 0, own = 0;
  for (size_t k : order) {
    const uint32_t c = counts[k];
    if (c < s.dense) continue;
    const uint32_t extra = pieces_beyond(s.per, c);
    CHECK(extra >= 1 && extra < kRefTilePieces);
    if (halo) {
      const uint32_t slot = taken;
      taken += extra + 1;
      if (slot + extra >= s.parts) continue;  // runs whole
    }
    listed += extra;
    own += k < (size_t)ntiles;
    uint32_t next = 1000;  // pieces 0 .. extra cover [1000, 1000 + c) in order
    for (uint32_t i = 0; i <= extra; ++i) {
      uint32_t beg = 1000, end = 1000 + c;
      piece_range(s.per, i, beg, end);
      CHECK(beg == next && end > beg && end - beg >= s.per);
      if (extra + 1 < kRefTilePieces) CHECK(end - beg < 2 * s.per);
      next = end;
    }
    CHECK(next == 1000 + c);
  }
  CHECK(listed <= s.max);
  CHECK(own <= kRefPieces / 2);
  return 0;
}

int main(int argc, char** argv) {
  std::mt19937 rng((unsigned)std::atoi(argc > 1 ? argv[1] : "0"));
  for (int it = 0; it < 400; ++it) {
    const long np = 65536 + (long)(std::exp2((double)(rng() % 13000) / 1000.0) * 65536) - 65536;
    const long ntiles = 1L << (rng() % 16);
    for (bool halo : {false, true}) {
      std::vector<uint32_t> counts(2 * ntiles, 0);
      // own entries: np in all, some keys crowded; halo entries: up to 7 np
      auto fill = [&](size_t first, long total) {
        const int crowds = (int)(rng() % 600);
        for (int q = 0; q < crowds && total > 0; ++q) {
          const long c = std::min<long>(total, rng() % 3 ? rng() % 30000 : rng() % (np + 1));
          counts[first + rng() % ntiles] += (uint32_t)c;
          total -= c;
        }
        counts[first + rng() % ntiles] += (uint32_t)(rng() % 2 ? total : 0);
      };
      fill(0, np);
      if (halo) fill(ntiles, 7 * np);
      if (check(np, ntiles, halo, counts, rng)) return 1;
    }
    // every key exactly at a limit
    const PieceSizes s = piece_sizes(np, ntiles, true);
    for (uint32_t c : {s.dense - 1, s.dense, 3 * s.per - 1, 3 * s.per, kRefTilePieces * s.per - 1, kRefTilePieces * s.per,
                       kRefTilePieces * s.per + 1}) {
      std::vector<uint32_t> counts(2 * ntiles, 0);
      for (long total = 8 * np, k = 0; k < 2 * ntiles && total >= c && (k < ntiles ? (k + 1) * (long)c <= np : true);
           ++k, total -= c)
        counts[k] = c;
      if (check(np, ntiles, true, counts, rng)) return 1;
    }
  }
  std::printf("ok\n");
  return 0;
}
