// tile_map.hpp -- work-item id -> (tile row, tile column, k-split) of the tile kernels.
//
// Plain C++ (no HIP header): the kernels include it through gemm_tn.hpp, and a host-only build
// under the address / undefined-behaviour sanitizers walks every id of a sweep of problems.
#pragma once

#if defined(__HIPCC__)
#define MJ_HD __host__ __device__ inline
#else
#define MJ_HD inline
#endif

namespace mj {

// Maps a linear work-item id to a tile (and a k-split).  The tiles of one k-split are put in a row: the
// grid of tiles is cut into strips -- at most kTall tile rows each, walked along N (n_first), or at most kLong
// tile columns each, walked along M -- and inside a strip the tiles that lie across it come one after the
// other, so any 32 consecutive tiles are a block of about 4 x 8 (the shape with the fewest operand panels)
// that shares its operand slices in an L2.  The k-splits follow each other in the same list; where one has fewer
// than 32 tiles, a group spans several.  Groups of 32 consecutive items go to
// the eight XCDs in turn (ids congruent mod 8 run on the same XCD): an XCD works on one such block at
// a time, the eight XCDs on eight neighbouring ones.
//
// The last, partial round (dealt()): in lots of 32 its tiles are work for a few XCDs while the others idle, an
// eighth each uses all of them.  That is better behind up to four full rounds, with 48 to 192 tiles left: logits of
// 246 x 3064, one round and 72, 128, 192 tiles 179 -> 169 us, 181 -> 171, 188 -> 182; of 507 x 2088, two rounds and
// 72 174.5 -> 166, four 290 -> 285.  Behind more rounds the XCDs have drifted apart, and the lots let the late
// ones off: eight rounds and 72 521 us in lots, 533 in eighths, 32 rounds 1996 and 2021.  So do 36 tiles (two rounds:
// 163 and 165), and a round that is nearly full has nothing to gain (242 tiles: 197 and 201).
//
// The list holds real tiles only and the strips of a grid differ by at most one in width, which
// is what keeps the XCDs equally loaded: with fixed 4 x 8 blocks and the empty slots of ragged ones as
// ids of their own, a grid of 9 tile columns walked along N gave every second block one live column out
// of eight, all of those on the same four XCDs (2049 tokens x 4096 x 128256: logits 2.9 ms against
// 1.85 ms in this order).
struct TileMap {
  static constexpr int kTall = 4, kLong = 8;
  int tiles_m, tiles_n, n_first, splits;
  int width, wide;         // strips: the first `wide` ones are width + 1 tiles across, the others `width`
  MJ_HD TileMap(int tm, int tn, int n_first_, int splits_)
      : tiles_m(tm), tiles_n(tn), n_first(n_first_), splits(splits_) {
    const int across = n_first ? tm : tn, most = n_first ? kTall : kLong;
    const int strips = across > 0 ? (across + most - 1) / most : 1;
    width = across / strips;
    wide = across - width * strips;
  }
  // whether the `left` tiles behind `round` full rounds are dealt evenly
  MJ_HD static bool dealt(int round, int left) { return left <= 192 && (round == 0 || (round <= 4 && left > 48)); }
  MJ_HD int tiles() const { return tiles_m * tiles_n * splits; }
  MJ_HD int items() const { return (tiles() + 255) & ~255; }
  MJ_HD bool tile(int pid, int& tm, int& tn, int& split) const {
    const int q = pid >> 3, xcd = pid & 7, round = q >> 5, within = q & 31;
    int at = (round << 8) + xcd * 32 + within;                  // place in the list of tiles
    const int left = tiles() - (round << 8);
    if (left <= 0) return false;
    if (dealt(round, left)) {                                   // the last round: an eighth each
      const int each = left >> 3, more = left & 7;
      if (within >= each + (xcd < more ? 1 : 0)) return false;
      at = (round << 8) + xcd * each + (xcd < more ? xcd : more) + within;
    } else if (at >= tiles()) {
      return false;
    }
    const int per = tiles_m * tiles_n, along = n_first ? tiles_n : tiles_m;
    split = at / per;
    at -= split * per;
    const int in_wide = wide * (width + 1) * along;
    int w = width, first = 0;                                   // width and first tile row / column of the strip
    if (at < in_wide) {
      w = width + 1;
    } else {
      at -= in_wide;
      first = wide * (width + 1);
    }
    const int strip = at / (w * along);
    at -= strip * w * along;
    const int step = at / w;
    const int x = first + strip * w + (at - step * w);
    tm = n_first ? x : step;
    tn = n_first ? step : x;
    return true;
  }
};

// The columns of the sampler's logits product: whole units, spread evenly over the work items (the first ones
// take one unit more where it does not come out even).
constexpr int kRowUnit = 32;
struct RowItems {
  int unit, units, items;
  MJ_HD RowItems(int vocab = 0, int items_ = 0, int unit_ = kRowUnit)
      : unit(unit_), units((vocab + unit_ - 1) / unit_), items(items_ < units ? items_ : units) {}
  MJ_HD int first(int item) const {       // first column of the item; the last item ends at the vocabulary's end
    const int base = units / items, wide = units - base * items;
    return (item * base + (item < wide ? item : wide)) * unit;
  }
};

}  // namespace mj
