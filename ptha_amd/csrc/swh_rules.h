// Rules that choose between two routes to the same result, from sizes alone (no device code).
#pragma once
#include <algorithm>

namespace swh {

constexpr int kSupTE = 64, kSupTN = 64;   // events and columns per tile of the dense event product
constexpr int kSupChunk = 16;             // samples per workgroup of its maxima

// lanes per event of the event lists' kernel (0: the sources' rows do not fit in LDS)
inline int list_lanes(int nsrc)
{
    const long long lds = 160 * 1024;
    return (nsrc + 1LL) * 256 <= lds ? 16 : (nsrc + 1LL) * 128 <= lds ? 8 : 0;
}

// Whether n_events events over ng gauges and 'samples' samples, which name 'entries' sources in
// all, are summed from lists of their sources or by the dense product over all nsrc sources.
// The expected kernel times (ms) decide:
//  - dense: its workgroups' time goes with the sources, and many rounds of workgroups (maxima:
//    about 430 resident) follow one another;
//  - lists: a workgroup stages its tile of all sources; each event then costs a tile its record
//    and (maxima) the maximum in memory, about as much as 100 of its sources, and its sources.
// With few sources the dense product thus wins however few of them an event names, and with many
// the lists, up to a share of them: 0.7, or 0.4 with weights, which are loaded per entry.
// Measured, dense / lists, in ms: maxima of 4096 events, 64 gauges, 100 samples, share 0.3: 10
// sources 0.063 / 0.27, 30 0.14 / 0.30, 50 0.20 / 0.30, 75 0.31 / 0.30, 512 1.8 / 0.35; 1000
// events: 20 sources 0.070 / 0.108, 30 0.10 / 0.10; 16 events, 30 sources, 300 samples 0.096 /
// 0.026. Series of 300 events, 64 gauges, 100 samples: 512 sources, share 0.5 0.32 / 0.21, 1000
// sources 0.56 / 0.44, weighted share 0.38 0.55 / 0.60; 128 events, 10 sources 0.0108 / 0.0138. Of
// 1583 such calls (10 to 1279 sources, 1 to 4096 events, 5 to 200 gauges) 11 lose more than a
// tenth to the other route, at most a third.
inline bool superpose_lists_fit(int nsrc, int ng, long long samples, long long n_events, long long entries,
                                bool weights, bool maxima)
{
    const int L = list_lanes(nsrc);
    if (!L) return false;
    const auto tiles = [](double n, int t) { return (double)(long long)((n + t - 1) / t); };
    const double E = (double)n_events, erows = tiles(E, kSupTE), K = tiles(nsrc, 4) * 4;
    if ((double)entries >= (weights ? 0.4 : 0.7) * erows * kSupTE * nsrc) return false;
    double dense, lists;
    const bool wide = L == 16;
    const double entry = (wide ? 3e-9 : 2.2e-9) * (double)entries;
    if (maxima) {
        const double rounds = std::max(1.0, tiles(ng, kSupTN) * erows * tiles((double)samples, kSupChunk) / 430.0);
        dense = 0.006 + 0.0036 * K * std::min(1.0, (double)samples / kSupChunk) * rounds;
        const double t = tiles(ng, L) * tiles((double)samples, 2);
        lists = 0.012 + 0.03 * std::min(1.0, E * t / 2e5) +
                t * (E * (wide ? 2.3e-7 : 1.8e-7) + entry * (weights ? 2.0 : 1.0));
    } else {
        const double N = (double)samples * 3 * ng;
        dense = 0.005 + K * (0.00015 + 3.6e-7 * tiles(N, kSupTN) * erows);
        lists = 0.0055 + nsrc * N * 8 / 5e9 +
                tiles(N, 2 * L) * (E * (wide ? 7e-8 : 4e-8) + entry * (weights ? 1.8 : 1.0));
    }
    return lists < dense;
}

// How many fused launches of three leapfrog steps have to follow one another on a single grid
// to be begun: the last one's boundary-flux sums cost a launch of their own (8 us), and each
// launch gains less than that over what it replaces where the grid is small. 'simple': truely
// linear without friction, whose rows are the shortest; 'due': max_stage after every step (it
// replaces three single steps, else one and a half pairs); 'odd': an odd number of launches in a
// stretch of an odd number of steps (to the call's end or the next update of max_U), of which pairs
// would leave a single step, which costs more than half a pair. In an even stretch a lone launch
// would leave such a step itself. Gain per launch in us, FP64 / FP32, max_stage not due: 8 x 6
// simple 1.6 / 1.6; 150 x 150 3.7 / 5.2, friction 3.4 / 6.1; 400 x 400 5.2 / 7.0, 1.0 / 6.7;
// 1024 x 1024 6.4 / 5.2, 3.8 / -0.2; 2048 x 2048 18 / 15, 31 / 10. Due: 8 x 6 3.7 / 3.7,
// 0.7 / 1.3; 150 x 150 4.0 / 5.2, 1.3 / 3.1; 400 x 400 12 / 9.4, 5.2 / 6.1; 700 x 500 19 / 17,
// 13 / 14.
constexpr int kFusedRunMost = 5;   // the most that is asked for

inline int fused_least_run(long long cells, bool simple, bool fp64, bool due, bool odd)
{
    if (due) {
        if (cells >= 300000) return 1;
        if (cells >= 100000) return simple ? 1 : 2;
        return simple || (!fp64 && cells >= 10000) ? 2 : 5;
    }
    if (odd && cells >= 300000) return 1;
    if (cells >= 3000000) return 2;
    if (simple) return cells >= 100000 ? 2 : cells >= 10000 ? 3 : 4;
    if (fp64) return cells >= 300000 ? 3 : 5;
    return cells >= 10000 && cells < 800000 ? 2 : 5;
}

}  // namespace swh
