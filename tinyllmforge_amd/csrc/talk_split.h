// Cutting the key ranges of row tiles (talk_prefill.hip).  Weights are complete before they are mixed, so parts of a row tile's keys add up.
//
// A row tile of `tq` rows walks `talk_steps` key tiles of 32.  One that walks more than `per` of them is cut: its extra parts have `per` steps
// each, from the first key on, and the rest, which ends on the diagonal, stays with the tile.
#pragma once
#include <stdint.h>

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

// Whether that pays, with `rows` rows in all portions: not
// - where no tile is longer than what the parts take, 1.2 even shares and six steps (16 heads, the layer, cut / whole, us: 24 portions of 250 tokens
//   93 / 89, 48 of 128 79 / 72, the same behind 1024 keys 272 / 251, but 12 of 400 99 / 106);
// - with row tiles of 16 rows (more than 16 heads) where nearly all places of the plan are taken and portions are long: a step of the kernel that
//   goes through the list takes 14 % longer there (one of 8000 1530 / 1421, four of 2048 483 / 449, three of 2600 565 / 535, but six of 1300
//   349 / 392, four of 1024 to 2048 347 / 375).
inline bool talk_cuts_pay(int64_t portions, int64_t tokens, int64_t rows, int64_t keys, int tq) {
  if (!talk_cuts(portions, tokens, keys, tq)) return false;
  const int64_t bound = (tokens + tq - 1) / tq * portions, tiles = rows / tq + (portions + 1) / 2 < bound ? rows / tq + (portions + 1) / 2 : bound;
  const int64_t longest = (keys + 31) / 32, before = keys > tokens ? (keys - tokens) / 32 : 0;
  if (tiles <= kTalkUnits && longest * 10 * 2 * kTalkUnits <= tiles * (longest + before) * 12 + 60 * 2 * kTalkUnits) return false;
  return tq > 16 || tiles <= 448 || tokens < 2048;
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
