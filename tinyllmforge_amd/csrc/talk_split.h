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
