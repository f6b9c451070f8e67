// The rules of the create-time races (opt-fft_amd/csrc/race.hpp) over a simulated clock:
// candidate i takes us[i] a launch; the first `slow` launches of it take `extra` more (clocks
// and buffers not yet warm), and every timed group may end late by a jitter of up to 4 us.
#include <cstdio>
#include <cstdlib>

#include "race.hpp"

using namespace fx;

struct Sim {
    std::vector<double> us, extra;
    std::vector<int> slow, fails_at;   // fails_at: launch number that fails, -1 none
    std::vector<int> done;
    double jitter = 0.0, spent = 0.0;
    unsigned seed = 1;
    int launches = 0;

    explicit Sim(std::vector<double> u) : us(u), extra(u.size(), 0.0), slow(u.size(), 0),
                                          fails_at(u.size(), -1), done(u.size(), 0) {}
    double uniform() { return (seed = seed * 1664525u + 1013904223u) / 4294967296.0; }
    bool launch(size_t i, int n)
    {
        for (int k = 0; k < n; ++k, ++done[i], ++launches) {
            if (done[i] == fails_at[i]) return false;
            spent += us[i] + (done[i] < slow[i] ? extra[i] : 0.0);
        }
        return true;
    }
    int race(const RaceRules& rules, int cycle)
    {
        std::vector<Trial> ts(us.size());
        auto go = [&](size_t i, int n) { return launch(i, n); };
        run_trials(ts, rules, cycle, go, [&](const std::vector<Trial>& c, std::vector<double>& t) {
            t.assign(c.size(), -1.0);
            bool any = false;
            for (size_t i = 0; i < c.size(); ++i) {
                if (!c[i].n) continue;
                const bool warm = launch(i, c[i].warm);
                const double start = spent;
                if (warm && launch(i, c[i].n))
                    t[i] = (spent - start + jitter * uniform()) * 1e-6 / c[i].n;
                any = true;
            }
            return any;
        });
        return race_winner(ts);
    }
};

#define CHECK(cond)                                                   \
    do {                                                              \
        if (!(cond)) {                                                \
            printf("FAIL line %d: %s\n", __LINE__, #cond);            \
            return 1;                                                 \
        }                                                             \
    } while (0)

int main()
{
    for (const RaceRules* r : {&kPlanRace, &kMultiRace}) {
        // A preset ten percent ahead wins however late its first launches are: three times its time.
        for (unsigned seed = 1; seed <= 200; ++seed) {
            Sim s({7.0, 7.2, 6.3, 7.1, 9.0});
            s.slow[2] = r->warmup + r->first;
            s.extra[2] = 14.0;
            s.jitter = 4.0;
            s.seed = seed;
            CHECK(s.race(*r, r == &kMultiRace ? 16 : 0) == 2);
        }
        // Near ties stay with the earlier registered one, 3% goes to the faster.
        Sim tie({100.0, 99.0, 101.0});
        CHECK(tie.race(*r, r == &kMultiRace ? 16 : 0) == 0);
        Sim ahead({100.0, 97.0, 101.0});
        CHECK(ahead.race(*r, r == &kMultiRace ? 16 : 0) == 1);
        // A kernel that does not launch, or stops launching, does not win and ends nothing.
        Sim fail({5.0, 10.0, 6.0});
        fail.fails_at = {0, -1, 7};
        CHECK(fail.race(*r, r == &kMultiRace ? 16 : 0) == 1);
        Sim none({5.0, 5.0});
        none.fails_at = {0, 0};
        CHECK(none.race(*r, r == &kMultiRace ? 16 : 0) == -1);
    }
    // What a mixed plan's race may cost, microseconds of launches: seven presets of a mix of 256
    // MiB, eleven launches of each, is what it cost before presets were added (12.7 ms); now ten.
    Sim mix({165, 190, 175, 172, 188, 168, 166, 157, 163, 158});
    CHECK(mix.race(kMultiRace, 2) == 7);
    printf("large mix: %d launches, %.1f ms\n", mix.launches, mix.spent * 1e-3);
    CHECK(mix.spent <= 12.7e3);
    // Short memory: as many sets as fit, by halves, with nothing kept of an attempt that failed.
    for (int room = 0; room <= 40; ++room) {
        int held = 0, tries = 0;
        const int got = fit_sets(16, [&](int n) {
            ++tries;
            held = n <= room ? n : 0;
            return held > 0;
        });
        int most = 16;
        while (most > room) most /= 2;
        CHECK(got == most && held == got && tries <= 5);
    }
    printf("OK\n");
    return 0;
}
