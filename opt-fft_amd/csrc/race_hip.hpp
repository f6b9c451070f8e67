// Rounds of a create-time race (race.hpp) timed with events.
#pragma once
#include <hip/hip_runtime.h>

#include "race.hpp"

namespace fx {

struct RaceEvents {
    std::vector<hipEvent_t> ev;   // two per candidate
    bool ok = true;

    explicit RaceEvents(size_t candidates)
    {
        ev.reserve(2 * candidates);
        for (size_t i = 0; i < 2 * candidates && ok; ++i) {
            hipEvent_t e;
            ok = hipEventCreate(&e) == hipSuccess;
            if (ok) ev.push_back(e);
        }
    }
    ~RaceEvents()
    {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    }
    RaceEvents(const RaceEvents&) = delete;
    RaceEvents& operator=(const RaceEvents&) = delete;

    // run_trials' round: the groups one after another on the stream, nothing waited for in between.
    template <class Launch>
    bool round(const std::vector<Trial>& ts, std::vector<double>& t, hipStream_t s, Launch launch)
    {
        t.assign(ts.size(), -1.0);
        size_t last = ts.size();
        for (size_t i = 0; i < ts.size(); ++i) {
            if (!ts[i].n) continue;
            const bool warm = launch(i, ts[i].warm);
            if (hipEventRecord(ev[2 * i], s) != hipSuccess) return false;
            if (warm && launch(i, ts[i].n)) t[i] = 0.0;
            if (hipEventRecord(ev[2 * i + 1], s) != hipSuccess) return false;
            last = i;
        }
        if (last == ts.size() || hipEventSynchronize(ev[2 * last + 1]) != hipSuccess) return false;
        for (size_t i = 0; i < ts.size(); ++i) {
            if (t[i] != 0.0) continue;
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, ev[2 * i], ev[2 * i + 1]) != hipSuccess) return false;
            t[i] = (double)ms * 1e-3 / ts[i].n;
        }
        return true;
    }
};

}  // namespace fx
