// Tile autotuner: the workgroup shape (elements per workgroup) of the
// Helmholtz kernels is chosen per (shape, operator, order, points,
// precision, geometry, input form) by timing every instantiated tile on
// the caller's own data, and remembered for the rest of the process so
// later operators of the same kind start from the measured choice, if they
// are not much larger than what was measured.
#pragma once

#include <functional>
#include <vector>

#include <hip/hip_runtime.h>

namespace nektar_amd {

struct TuneKey {
    int shape, op, nm, nq, fp32, deformed, form;  // form 0: element-local input, 1: gathered from a C0 vector
    bool operator<(const TuneKey &o) const;
};

// The choice measured on nelmt elements or the next larger count, else on the
// largest one if nelmt is at most kTunedReach times that; 0 when there is none.
// What wins on a collection that leaves CUs idle can lose on one that does not:
// chosen on 64 elements and run on some 10 M coefficients, affine hexes at
// NM = 3 and 6 take 1.2 times the default's time, curved ones, FP64 at NM = 8
// 1.4 times and FP32 at NM = 5 1.6 times.
constexpr int kTunedReach = 4;
int tuned_tile(const TuneKey &k, int nelmt);
void record_tile(const TuneKey &k, int nelmt, int tile);
void clear_tuned_tiles();

// Times launch(tile) for every candidate (warm-up, then `reps` launches
// between two events on `s`, again for those near the fastest: tune_pick.hpp)
// and returns the fastest tile; the shortest mean time of each candidate in
// microseconds goes to times_us when given.  A candidate whose launch fails is
// skipped.
int time_tiles(hipStream_t s, const std::vector<int> &candidates, const std::function<hipError_t(int)> &launch,
               int reps, std::vector<double> *times_us = nullptr);

}  // namespace nektar_amd
