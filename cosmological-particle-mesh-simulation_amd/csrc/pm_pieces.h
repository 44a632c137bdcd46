// Pieces of crowded tiles: the arithmetic of their sizes, for the scan that lists them and the kernels that
// take them (plain C++, constexpr so that both sides of a kernel launch use it).
//
// A key (own or halo segment of a tile's entries) of at least `dense` entries is cut into pieces of `per` (64
// longer ones at most): the tile's block takes the first, the others are listed by the scan and shared out
// to further blocks.  The deposit's blocks of one tile leave FP64 partial sums; the last to do so (ticket)
// adds them up, about 1 us each, and rounds.
// per is 4096 entries, four batches of a deposit block (about 15 us, what the meeting of a tile's blocks
// costs), or N_p / 512: at most 256 tiles have own pieces, and a block's share of a call stays small.
// dense is 2 per, and on 64 tiles or more twice their mean: evenly filled, they keep the chip busy by
// themselves (density of 2.1 M random particles on 96^3, whole / in pieces of 4096: 248 / 336 us; on
// 48^3, 27 tiles, 650 / 429).  Keys beyond the room for partial sums run whole.
#pragma once
#include <cstdint>

namespace pm {

constexpr long kRefPiece = 4096, kRefPieces = 512;
constexpr uint32_t kRefTilePieces = 64;  // of one key

struct PieceSizes {
  uint32_t per = 0, dense = 0;
  uint32_t max = 0;    // listed pieces at most: a piece beyond its key's first holds >= per entries
  uint32_t parts = 0;  // partial sums of the deposit (the push needs none)
};
// halo: own and halo keys, up to 8 entries a particle (the deposit); otherwise own ones
constexpr PieceSizes piece_sizes(long np, long ntiles, bool halo) {
  PieceSizes s{};
  const long per = (np + kRefPieces - 1) / kRefPieces;
  s.per = (uint32_t)(per > kRefPiece ? per : kRefPiece);
  const long mean2 = ntiles >= 64 ? 2 * np / ntiles : 0;
  s.dense = (uint32_t)(mean2 > 2L * s.per ? mean2 : 2L * s.per);
  s.max = (uint32_t)((halo ? 8 : 1) * np / s.per);
  if (halo) s.parts = s.max < 2 * kRefPieces ? s.max : (uint32_t)(2 * kRefPieces);
  return s;
}

// pieces of a dense key beyond its first
constexpr uint32_t pieces_beyond(uint32_t per, uint32_t count) {
  const uint32_t n = count / per;
  return (n < kRefTilePieces ? n : kRefTilePieces) - 1;
}
// narrows the entries [beg, end) of a dense key to its piece i (0: what the tile's own block takes)
constexpr void piece_range(uint32_t per, uint32_t i, uint32_t& beg, uint32_t& end) {
  const uint32_t last = pieces_beyond(per, end - beg), len = (end - beg) / (last + 1);
  beg += i * len;
  if (i < last) end = beg + len;
}

}  // namespace pm
