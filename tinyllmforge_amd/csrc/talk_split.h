// Cutting the key ranges of row tiles (talk_prefill.hip).  Weights are complete before they are mixed, so parts of a row tile's keys add up.
//
// A row tile of `tq` rows walks `talk_steps` key tiles of 32.  One that walks more than `per` of them is cut: its extra parts have `per` steps
// each, from the first key on, and the rest, which ends on the diagonal, stays with the tile.
#pragma once
#include <stdint.h>

#include "prompt_tiles.h"

namespace tlf {

constexpr int kTalkUnits = 256;     // compute units, each with one workgroup
constexpr int kTalkTiles = 512;     // row tiles of a launch that cuts them, at most
constexpr int kTalkExtras = 256;    // their extra parts, at most: each takes an even share of all steps, or more
constexpr int kTalkLeast = 3;       // steps of a part at least

// Whether tiles are cut: `portions` of up to `tokens` rows, contexts of up to `keys`.  With fewer tiles than units a launch is as long as its
// longest tile (16 heads: one portion of 130 tokens behind 2048 keys 308 -> 42 us, one of 700 109 -> 38, of 5000 702 -> 296); with more, where
// lengths differ much (eight of 1061 to 2048 tokens 312 -> 261, 20 of 300 to 600 126 -> 101; 32 heads, four of 626 to 1251 198 -> 180).
// Not so many portions of a few hundred tokens: their tiles are alike, and whole ones stay on the XCD that has read their keys (32 heads, 16 of
// 150 to 300 59 us whole, 70 cut; 16 heads, 60 of 90 to 180 42 and 51).
__host__ __device__ inline bool talk_cuts(int64_t portions, int64_t tokens, int64_t keys, int tq) {
  const int64_t tiles = (tokens + tq - 1) / tq * portions;
  return keys > kTalkLeast * 32 && (tiles <= 192 || (tiles <= kTalkTiles && tokens >= 512));
}

// What a launch has to do, as the host knows it: portions, the most tokens of one, their rows, the keys that rows see summed over rows (0: not
// known), the most keys of a portion.
struct TalkLoad {
  int64_t portions, tokens, rows, reads, keys;
};
// Row tiles, and the key tiles that they walk.
inline int64_t talk_bound(const TalkLoad &l, int tq) { return (l.tokens + tq - 1) / tq * l.portions; }
inline int64_t talk_real_tiles(const TalkLoad &l, int tq) {
  const int64_t bound = talk_bound(l, tq), even = l.rows / tq + (l.portions + 1) / 2, tiles = even > l.portions ? even : l.portions;
  return tiles < bound ? tiles : bound;
}
inline double talk_all_steps(const TalkLoad &l, int tq) {
  const int64_t longest = (l.keys + 31) / 32, before = l.keys > l.tokens ? (l.keys - l.tokens) / 32 : 0;
  return talk_real_tiles(l, tq) * (l.reads > 0 && l.rows > 0 ? static_cast<double>(l.reads) / (32.0 * l.rows) + 0.5 : 0.5 * (longest + before));
}

// Whether that pays: not where no tile is longer than what the parts take, 1.2 even shares and six steps (16 heads, the layer, cut / whole, us: 24
// portions of 250 tokens 93 / 89, 48 of 128 79 / 72, the same behind 1024 keys 272 / 251, but 12 of 400 99 / 106).
//
// With more tiles than units, whole ones take an even share or the longest, whichever is more, and with row tiles of 16 rows (more than 16 heads) a
// step of the kernel that goes through the list takes 14 % longer: one of 8000 1530 / 1421, four of 2048 483 / 449, eight of 600 behind 1024
// keys 484 / 448, but four of 1024 to 2048 347 / 375.  An XCD takes whole portions four at a time (prompt_tiles.h); where one or two are left for the
// end, and the others fill the chip, their longest tiles begin late: five of 1500 419 / 506, six of 1300 388 / 422, but seven of 800 227 / 199.
inline bool talk_cuts_pay(const TalkLoad &l, int tq) {
  if (!talk_cuts(l.portions, l.tokens, l.keys, tq)) return false;
  const int64_t tiles = talk_real_tiles(l, tq);
  const double share = talk_all_steps(l, tq) / kTalkUnits, longest = static_cast<double>((l.keys + 31) / 32);
  if (tiles <= kTalkUnits) return longest > 1.2 * share + 6;
  if (tq > 16) return true;
  PromptTiles t;
  prompt_tiles_make(t, (l.tokens + tq - 1) / tq, 1, l.portions);
  const int last = t.per_xcd % t.together;
  const bool late = t.per_xcd > t.together && (last == 1 || last == 2) && tiles * (t.per_xcd - last) > static_cast<int64_t>(kTalkUnits) * t.per_xcd;
  return 1.2 * share + 6 < (longest > share ? longest : share) * (late ? 1.5 : 1);
}

// How the short portions of a step run: row by row, in one launch with the long ones, or in one of their own.  Every portion of a launch has
// workgroups for the row tiles of the longest.  From 64 short rows on (fewer: row by row) whichever takes least by these estimates, in us, of
// the rows' kernels and of a launch of row tiles.  Against the measured best of the three on 314 steps of 16 and 32 heads, 1 to 200 short portions of 2 to 127
// tokens behind up to 4096, up to 60 long ones of up to 8000, up to 400 single tokens: all together 1.7 % more, 1.29 x in one step at
// most; row by row always 18 % (5.2 x), one launch always 75 % (11.8 x).
enum TalkRoute { kTalkByRows, kTalkTogether, kTalkApart };
inline double talk_rows_us(const TalkLoad &l, bool singles) {        // with single tokens the kernels run anyway
  return (singles ? 0 : 12) + 0.8e-3 * l.reads + 0.05 * l.rows + (singles ? 0.0045 : 0.0055) * l.keys;
}
inline double talk_tiles_us(const TalkLoad &l, int heads, int tq) {
  if (l.portions == 0) return 0;
  const double step = 5.2, share = talk_all_steps(l, tq) / kTalkUnits, longest = l.keys / 32.0;
  const double stats = 0.0285 * l.keys + 2.4e-7 * heads * l.reads;
  if (talk_cuts_pay(l, tq)) return 25 + stats + step * (1.5 * share + 3 < longest ? 1.5 * share + 3 : longest);
  const int64_t tiles = talk_real_tiles(l, tq), empty = talk_bound(l, tq) - (tiles > kTalkUnits ? tiles : kTalkUnits);
  return 10 + stats + step * (1.4 * share > longest ? 1.4 * share : longest) + (empty > 0 ? 0.1 * empty : 0);
}
inline TalkRoute talk_route(bool singles, const TalkLoad &s, const TalkLoad &l, int heads, int tq) {
  if (s.rows < 64) return kTalkByRows;
  const TalkLoad both{s.portions + l.portions, s.tokens > l.tokens ? s.tokens : l.tokens, s.rows + l.rows, s.reads + l.reads, s.keys > l.keys ? s.keys : l.keys};
  const double beside = talk_tiles_us(l, heads, tq), rows = talk_rows_us(s, singles) + beside, apart = talk_tiles_us(s, heads, tq) + beside;
  const double together = l.portions ? talk_tiles_us(both, heads, tq) : apart;
  return rows < together && rows < apart ? kTalkByRows : together <= apart ? kTalkTogether : kTalkApart;
}

__host__ __device__ inline int talk_tiles(int tokens, int tq) { return tokens <= 0 ? 0 : (tokens - 1) / tq + 1; }
__host__ __device__ inline int talk_steps(int start, int tokens, int tq, int x) {
  const int end = tokens - x * tq < tq ? tokens : (x + 1) * tq;
  return (start + end - 1) / 32 + 1;
}
__host__ __device__ inline int talk_extras(int steps, int per) { return (steps - 1) / per; }

// Steps of a part: an even share of all steps.  The longest parts are taken first, and what is left of tiles evens out the rest (16 heads, one
// portion of 5000 tokens: 5/4 of a share 321 us, 3/4 389, this 281).  A few more steps where each tile and part then has a unit of its own: a
// unit's second part begins with latency of about four steps.  extras(per): extra parts of all tiles.
template <class Extras>
__host__ __device__ inline int talk_per(int64_t steps, int tiles, Extras extras) {
  const int64_t even = (steps + kTalkUnits - 1) / kTalkUnits;
  const int share = even < kTalkLeast ? kTalkLeast : even < 1 << 26 ? static_cast<int>(even) : 1 << 26;
  for (int per = share; per <= share + 4; ++per)
    if (tiles + extras(per) <= kTalkUnits) return per;
  return share;
}

// 128 classes of length, the longest first.
__host__ __device__ inline int talk_class(int steps, int per) { return steps >= per ? 0 : 127 - static_cast<int>(static_cast<int64_t>(steps) * 127 / per); }

}  // namespace tlf
