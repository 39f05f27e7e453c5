// pdt_tune.hpp -- tile-shape cache of the autotuner.
//
// Tiles are keyed by the problem shape; values are the coils per LDS chunk
// of the forward (cb) and adjoint (cb_a) row kernels, the columns per group
// (cg) of the column kernel, the rows per item (rpi) of the denoising
// kernels and the occupancy caps (workgroups per CU) of the forward row,
// column, adjoint row and denoising passes.  A value of 0 means "use the
// built-in default" (no cap, for the occupancy, and two launches per MRI
// iteration where possible).  The cache is process-wide and, when the environment
// variable PDT_TUNE_CACHE names a file, loaded from / saved to that file, so a
// tuned choice is deterministic across runs.
#pragma once

#include <string>

namespace pdt {

struct TuneKey {
  int kind, dt, W, H, Hk, C, nc, ns;
  bool operator<(const TuneKey& o) const;
  std::string str() const;
};

struct TuneVal {
  int cb = 0, cg = 0, rpi = 0, cb_a = 0;
  int wpc[4] = {0, 0, 0, 0};  // workgroups per CU of the passes (0: no cap)
  int tb[3] = {0, 0, -1};     // temporally blocked ROF tiles x, y, iterations (-1: default, 0: off)
  int dual_px = 0;            // TGV denoising dual step: pixels per thread (0: default)
  int unpaired = 0;           // MRI: three launches per iteration even where two would do
};

TuneVal tune_lookup(const TuneKey& k);
// Whether a choice is stored for k.
bool tune_has(const TuneKey& k);
void tune_store(const TuneKey& k, const TuneVal& v);

// A slice of a batch of operator solvers: its transform lengths, million
// sensitivities on half the k-space grid (C W Hk / 2; 4 times in double
// precision, whose passes take that much longer per element) and whether it
// would run paired iterations alone.
struct BatchSlice {
  int W, Hk;
  double x;
  bool paired;
};
// Whether n slices are faster as single solves on a few streams than as one
// work-list launch per pass and group of equal transform lengths.  A group's
// launches follow one another, each with its own tail, and stream every slice
// through DRAM; single solves overlap, pair their iterations where they can and
// keep fewer slices in the caches, but pay every chunk's start per slice, and
// three or more of them take 4 ms per 100 iterations however small they are.
// Fitted to 378 batches of 2 to 32 slices (48 x 48 to 384 x 384, 1 to 15 coils,
// up to four sizes, all three operators, both precisions), both ways measured
// over 100 iterations: the way it takes is within 1 % of the faster one in the
// mean and 11 % at the worst, and at the worst 4 % slower than the work lists.
// On either side of the line: 8 slices of 320 x 320, 15 coils 21.3 ms batched
// and 14.7 as singles; 2 of 48 x 48 and 64 x 64, 6 coils 5.3 and 2.2; 8 of 64 x
// 64, 15 coils 4.4 and 7.5; 3 of 128 x 128, 4 coils 2.7 and 3.9.
bool batch_singles_faster(const BatchSlice* s, int n);

}  // namespace pdt
