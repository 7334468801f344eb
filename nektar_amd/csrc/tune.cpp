#include "tune.hpp"

#include <cstdint>
#include <map>
#include <mutex>
#include <tuple>

#include "common.hpp"
#include "tune_pick.hpp"

namespace nektar_amd {

bool TuneKey::operator<(const TuneKey &o) const
{
    return std::tie(shape, op, nm, nq, fp32, deformed, form) <
           std::tie(o.shape, o.op, o.nm, o.nq, o.fp32, o.deformed, o.form);
}

namespace {
std::mutex g_tune_mutex;
// by the element count of the measurement
std::map<TuneKey, std::map<int, int>> &tune_table()
{
    static std::map<TuneKey, std::map<int, int>> t;
    return t;
}
}  // namespace

int tuned_tile(const TuneKey &k, int nelmt)
{
    std::lock_guard<std::mutex> l(g_tune_mutex);
    auto it = tune_table().find(k);
    if (it == tune_table().end()) return 0;
    const auto &by_count = it->second;
    const auto larger = by_count.lower_bound(nelmt);
    if (larger != by_count.end()) return larger->second;
    const auto &largest = *by_count.rbegin();
    return nelmt <= (int64_t)kTunedReach * largest.first ? largest.second : 0;
}

void record_tile(const TuneKey &k, int nelmt, int tile)
{
    std::lock_guard<std::mutex> l(g_tune_mutex);
    tune_table()[k][nelmt] = tile;
}

void clear_tuned_tiles()
{
    std::lock_guard<std::mutex> l(g_tune_mutex);
    tune_table().clear();
}

int time_tiles(hipStream_t s, const std::vector<int> &candidates, const std::function<hipError_t(int)> &launch,
               int reps, std::vector<double> *times_us)
{
    NMF_REQUIRE(!candidates.empty(), NMF_ERR_UNSUPPORTED, "no tile candidates");
    NMF_REQUIRE(reps > 0, NMF_ERR_INVALID, "reps must be positive");
    hipEvent_t e0, e1;
    NMF_HIP(hipEventCreate(&e0));
    NMF_HIP(hipEventCreate(&e1));
    const auto sample = [&](int t, int round) {
        // the first round is the one in which slow candidates take part
        const int n = round == 0 ? (reps + 1) / 2 : reps;
        if (launch(t) != hipSuccess) {
            (void)hipGetLastError();
            return -1.0;
        }
        NMF_HIP(hipEventRecord(e0, s));
        for (int r = 0; r < n; ++r) NMF_HIP(launch(t));
        NMF_HIP(hipEventRecord(e1, s));
        NMF_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        NMF_HIP(hipEventElapsedTime(&ms, e0, e1));
        return 1e3 * ms / n;
    };
    const int best = pick_tile(candidates, sample, times_us);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    NMF_REQUIRE(best > 0, NMF_ERR_DEVICE, "every tile candidate failed to launch");
    return best;
}

}  // namespace nektar_amd
