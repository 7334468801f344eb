// Choice among tile candidates from timings (host code, no HIP).
#pragma once

#include <algorithm>
#include <functional>
#include <limits>
#include <vector>

namespace nektar_amd {

// The candidate with the shortest sample, -1 if none can run.  sample(t, k) is
// timing k of t in us, negative if t cannot run.  A single timing of a short
// kernel is off by several per cent, and the first ones more (the clocks are
// still low), so every candidate within 1.25 of the shortest is timed again,
// kTuneRounds times in all and in turn, and the shortest counts; a tie goes to
// the earlier candidate.  15 kinds of hexes, 500 to 90,000 elements, tuned six
// times each: with one timing a choice up to 5 % slower than the default, with
// these up to 0.6 %.
constexpr int kTuneRounds = 3;
inline int pick_tile(const std::vector<int> &candidates, const std::function<double(int, int)> &sample,
                     std::vector<double> *times_us = nullptr)
{
    const double inf = std::numeric_limits<double>::infinity();
    std::vector<double> best(candidates.size(), inf);
    std::vector<bool> runs(candidates.size(), true);
    for (int round = 0; round < kTuneRounds; ++round) {
        const double limit = round == 0 ? inf : 1.25 * *std::min_element(best.begin(), best.end());
        for (size_t c = 0; c < candidates.size(); ++c) {
            if (!runs[c] || best[c] > limit) continue;
            const double us = sample(candidates[c], round);
            if (us < 0) runs[c] = false;
            else best[c] = std::min(best[c], us);
        }
    }
    if (times_us) *times_us = best;
    const auto it = std::min_element(best.begin(), best.end());
    return it == best.end() || *it == inf ? -1 : candidates[it - best.begin()];
}

}  // namespace nektar_amd
