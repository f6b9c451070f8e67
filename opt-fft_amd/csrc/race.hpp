// Create-time races: candidates timed in turn, in rounds of groups of launches, and dropped as
// the rounds show them behind.  Plain C++ over two callables, so that the rules run on the CPU
// too; race_hip.hpp times the groups with events.
#pragma once
#include <cstddef>
#include <vector>

namespace fx {

// One candidate, launched in groups of n between two events.
struct Trial {
    int n;        // launches per group; 0: failed to launch, or out of the race
    int warm;     // launches before a group that are not timed
    double best;  // fastest group of the rounds that count, seconds per launch
};

// One round: every candidate still in the race runs a group of about `group` seconds, least ..
// most launches; those slower than `keep` times the fastest are out.  anew: groups are sized
// from the times so far, which are then forgotten, and a third as many launches of the same
// kernel, or `cycle` (run_trials) if that is more, run before each, not timed.
struct RaceRound {
    double group;
    int least, most;
    bool anew;
    double keep;
};

struct RaceRules {
    int warmup, first;   // launches before and in the group that sizes the others
    RaceRound round[4];
    int nrounds;
};
// Plans (plan.cpp): groups of about 300 us, 1.5 ms in the final, as event timing jitter of a few
// microseconds would otherwise decide between kernels of ~10 us.  Timed one after the other
// instead of in turn, kernels 5% apart changed places from run to run.  A kernel's first launches
// run against what the kernel before it left in the caches: in groups of five a persistent 6^3
// complex128 kernel takes 74 us to a staged one's 77, and 79.5 to 77.6 in runs of 40; at 17^3 x
// 2798 the order of two turns round likewise (88 : 91 and 90 : 87).
constexpr RaceRules kPlanRace = {
    2, 5,
    {{300e-6, 5, 64, false, 1.25}, {300e-6, 5, 64, false, 1.10}, {1.5e-3, 5, 256, true, 1.05}, {1.5e-3, 5, 256, false, 1.05}},
    4};
// Mixed launches (multi_plan.cpp): a race that no record saves, over eleven presets of 100 us a
// launch at 256 MiB of input, so the groups are shorter.  All that count are timed behind a launch on
// every set of the buffers (`cycle`; one launch where they all fit in the 256 MB cache): the preset
// before leaves its lines there, written in part.  Right behind multi_c128_t192, multi_c128_t192_lin
// takes 97 us for 6^3 x 20000, 8^3 x 8000, 12^3 x 3000 and multi_c128_t192 itself 78; behind
// launches of their own 80 and 85.
constexpr RaceRules kMultiRace = {1, 1, {{100e-6, 2, 64, true, 1.04}, {150e-6, 2, 64, true, 1.03}}, 2};

// launch(i, n): n launches of candidate i, false if one failed.  round(ts, t): one group of every
// candidate with n > 0, seconds per launch into t (not positive where a launch failed), false
// if nothing could be timed.  Warm-up launches and a group of `first` size every candidate's
// groups (which also brings the clocks up); that group decides nothing: a few microseconds of
// event jitter or buffers not touched before are much of it.  Trials that end with best < 1e29
// have run to the end.
template <class Launch, class Round>
void run_trials(std::vector<Trial>& ts, const RaceRules& rules, int cycle, Launch launch, Round round)
{
    std::vector<double> t;
    auto size = [&](double per, const RaceRound& r) {
        const double n = r.group / per;
        return n < r.least ? r.least : n > r.most ? r.most : (int)n;
    };
    for (size_t i = 0; i < ts.size(); ++i) ts[i] = Trial{launch(i, rules.warmup) ? rules.first : 0, 0, 1e30};
    if (!round(ts, t)) return;
    for (size_t i = 0; i < ts.size(); ++i) {
        if (t[i] > 0) ts[i].best = t[i];
        else ts[i].n = 0;
    }
    for (int k = 0; k < rules.nrounds; ++k) {
        const RaceRound& r = rules.round[k];
        if (k == 0 || r.anew)
            for (Trial& c : ts) {
                if (!c.n) continue;
                c.n = size(c.best, r);
                if (r.anew) c.warm = c.n / 3 > cycle ? c.n / 3 : cycle;
                c.best = 1e30;
            }
        if (!round(ts, t)) return;
        double lead = 1e30;
        for (size_t i = 0; i < ts.size(); ++i) {
            if (!ts[i].n) continue;
            if (t[i] <= 0) ts[i].n = 0, ts[i].best = 1e30;
            else if (t[i] < ts[i].best) ts[i].best = t[i];
            if (ts[i].best < lead) lead = ts[i].best;
        }
        for (Trial& c : ts)
            if (c.best > r.keep * lead) c.n = 0, c.best = 1e30;
    }
}

// Sets of buffers that a race may use: alloc(n) for n = sets and then half as many each time, until
// it succeeds (it keeps nothing where it fails).  0 if not even one was had.
template <class Alloc>
int fit_sets(int sets, Alloc alloc)
{
    for (; sets >= 1; sets /= 2)
        if (alloc(sets)) return sets;
    return 0;
}

// The candidate a race picked, -1 if none ran to the end.  A later one must beat the incumbent by
// more than 1.5% (above the run-to-run spread of one trial) and a tenth of a microsecond more,
// so near-ties resolve the same way each time, to the earlier-registered variant.  The tenth is
// for kernels that last as long as a launch: there a full queue hides a kernel's start, which a
// paced caller pays (6^3 complex128 x 289: 3.74 us here to the staged kernel's 3.82, and 4.5 to
// 3.9 launched from Python).
inline int race_winner(const std::vector<Trial>& ts)
{
    int win = -1;
    for (size_t i = 0; i < ts.size(); ++i)
        if (ts[i].best < 1e29 && (win < 0 || ts[i].best < 0.985 * ts[win].best - 0.1e-6))
            win = (int)i;
    return win;
}

}  // namespace fx
