// Which (sequence, plane, row tile) of a batch of prompt portions a workgroup takes.  A plane is what shares keys: a KV head, or a
// pass over some of its query heads.
//
// Workgroup w runs on XCD w % 8, and each XCD has its own L2.  Portions have unequal lengths and a row tile's work grows with its
// place, so the planes of all sequences are dealt to the XCDs in turn.  Where there are few of them, or they do not come out even,
// each is cut into two, four or eight `parts`, its row tiles dealt to its parts in turn and the parts to the XCDs.  Which part gets the
// last tile turns each time the parts have gone once around the XCDs: otherwise eight parts are the eight XCDs, and the last tile of
// every sequence runs on the same one.  (Handing each XCD a run of consecutive (sequence, plane) pairs gives it whole sequences, and
// the launch waits for the XCD with the longest one.)
//
// No more parts than that: a plane's keys are read by as many XCDs as it has parts.  Mixed heads (one plane, 16 heads, talk_prefill.hip),
// parts 8 / 4 / 2 / 1: 64 prompts of 128 tokens 63 / 40 / 38 / 37 us, 30 of 151 to 300 82 / 77 / 59 / 58, eight of 1061 to 2048
// 328 / 321 / 352 / 356; 32 heads, 16 of 300 81 / 62 / 63 / 63, eight of 1061 to 2048 551 / 580 / 659 / 660.  So parts are added until every
// XCD has six of them, and as many as any other one or ten.
//
// An XCD takes its planes four at a time and walks their row tiles together, the last ones (the longest key ranges) first, so that
// it ends on short workgroups while the planes at work still fit its L2 (4 x 1 MB at 2048 keys of 2 x 128 bf16).  The order of the
// four turns by one from row tile to row tile: an XCD deals its workgroups to its four shader engines in turn as well, and without
// the turn each engine gets all row tiles of one sequence, and the launch waits for the engine with the longest.  (`together`: others
// than four, where tiles of a plane share more than keys.)
//
// Eight prompts of 1061 to 2048 tokens, 32 heads on 8 KV heads (sink_prefill.hip): 521 us with either of the two mistakes, as long
// as eight prompts of 2048; 355 us so.
#pragma once
#include <stdint.h>

namespace tlf {

struct PromptTiles {
  int32_t xtiles, planes, parts, per_part;   // row tiles; planes of a sequence; parts of a plane, their tiles
  int32_t all_parts, per_xcd, together;                // of all sequences; for an XCD, at most
};

// Workgroups to launch, 0: too many.
inline int prompt_tiles_make(PromptTiles &t, int64_t xtiles, int64_t planes, int64_t seqs, int together = 4) {
  int parts = 1;
  auto enough = [&](int64_t all) { return all >= 80 || (all >= 48 && all % 8 == 0); };
  while (parts < 8 && planes * parts % 8 && !enough(planes * parts * seqs)) parts *= 2;
  const int64_t most = 1 << 27, per_part = (xtiles + parts - 1) / parts, all_parts = planes * parts * seqs, per_xcd = (all_parts + 7) / 8;
  if (per_part > most || per_xcd > most || per_part * per_xcd > most) return 0;
  t = PromptTiles{static_cast<int32_t>(xtiles), static_cast<int32_t>(planes), parts, static_cast<int32_t>(per_part), static_cast<int32_t>(all_parts),
                  static_cast<int32_t>(per_xcd), together};
  return static_cast<int>(per_part * per_xcd * 8);
}

// The grid, in rows of 2^20: a dimension of a launch holds less than 2^32 threads, 2^23 workgroups of 512.
constexpr int kPromptRow = 1 << 20;
template <class Dim3>
Dim3 prompt_grid(int blocks) {
  return blocks <= kPromptRow ? Dim3(blocks) : Dim3(kPromptRow, (blocks + kPromptRow - 1) / kPromptRow);
}
__host__ __device__ inline int prompt_block(unsigned int x, unsigned int y) { return static_cast<int>(y * kPromptRow + x); }

// False: nothing to do.
__host__ __device__ inline bool prompt_tile(const PromptTiles &t, int block, int &seq, int &plane, int &xt) {
  const int i = block >> 3;
  if (i >= t.per_part * t.per_xcd) return false;
  const int first = i / (t.together * t.per_part) * t.together;
  const int together = t.per_xcd - first < t.together ? t.per_xcd - first : t.together, within = i - first * t.per_part;
  const int step = within / together, part = (first + (within + step) % together) * 8 + (block & 7), of_seq = t.planes * t.parts;
  seq = part / of_seq;
  plane = part % of_seq / t.parts;
  if (part >= t.all_parts) return false;
  xt = t.xtiles - 1 - (step * t.parts + (part % t.parts + (part >> 3)) % t.parts);
  return xt >= 0;
}

}  // namespace tlf
