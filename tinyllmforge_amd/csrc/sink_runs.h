// Which rows of a step the preparation of attention with sinks works on in runs (sink_prep_rows_kernel, sink_attn.hip).
#pragma once
#include <stdint.h>

namespace tlf {

// The first of these rows, n: none.  The step has n rows, the first `singles` of them single tokens, and `seqs` sequences in all (0: not known);
// hy: workgroups for a row's heads, 16 each.  All figures: us of the preparation, runs / four rows a workgroup, 32 + 2 x 8 heads (hy = 3) and
// 16 + 2 x 8 (hy = 2) of 128.
//
// Without a convolution rows do not depend on each other: what runs save is loading the weights (4000 rows 22.8 / 25.2 and 17.3 / 19.2).  Few rows do not fill
// the chip in runs (1500 rows, hy = 2 11.1 / 9.8), and many are bound by HBM (12000, hy = 3 73.6 / 70.4).
//
// With one, a run's sequences follow each other, each with loads that are waited for, and all their rows share those of the rows before.  So not
// - up to 3 x 1024 rows and workgroups, which are on the chip at once in fours (1500 rows, hy = 2 14.9 / 14.2; 1600 14.6 / 18.0);
// - portions of two or three tokens (4500 of two 101 / 87; of three 44.5 / 42.5 with 4000 rows, 77 / 88 with 9000), but of four (14.1 / 18.0 with 1100);
// - single tokens.  A few may lead the first run (two and 2000 rows 22 / 25.5, four and 3000 29.4 / 34.5, 27 / 24.6 with hy = 2); more get a launch of
//   their own where that is repaid (128 and 3000 36.7 / 38.7, with hy = 2 and 1500 20.8 / 18.8; in runs 50 and 35).
inline int64_t sink_runs_from(int64_t n, int64_t singles, int64_t seqs, int64_t hy, bool conv) {
  if (n <= 1024) return n;
  if (!conv) return n * hy >= 5 * 1024 && n * hy < 24 * 1024 ? 0 : n;
  const int64_t rows = n - singles, portions = seqs - singles;
  if (portions <= 0 || rows * hy <= 3 * 1024) return n;
  if (rows < portions * (rows * hy >= 16 * 1024 ? 3 : 4)) return n;
  if (singles <= 4 && n * hy >= singles * 2000) return 0;
  return rows * hy >= 10 * 1024 ? singles : n;
}

// Rows of a run: long ones save more, shorter ones make more workgroups, four for each compute unit at least with 24 and three with 16 (36,700 workgroups of a
// row: runs of 32 90 us, 24 84, 16 92, 8 106; 3400: 16 23, 8 19).
inline int sink_run_rows(int64_t rows, int64_t hy) { return rows * hy >= 24 * 1024 ? 24 : rows * hy >= 16 * 768 ? 16 : 8; }

}  // namespace tlf
