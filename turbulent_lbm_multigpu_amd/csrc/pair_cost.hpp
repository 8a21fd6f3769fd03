// pair_cost.hpp -- which step sequences run as fused pairs (pair_kernel): both
// ways' times as fitted to measurements, us on one device.  Plain C++: the
// choices are checked on the CPU.
#pragma once

#include <algorithm>
#include <array>
#include <functional>
#include <queue>
#include <utility>
#include <vector>

#include "pair_plan.hpp"

namespace lbm {

// Work-groups of the pair kernel that run at once: the LDS of one takes a compute unit.
constexpr long long kPairSlots = 256;

// A half-step in place of `cells` in all.  It moves 38 values a cell; past the
// last-level cache (256 MB) by what the cache no longer holds, which the
// non-temporal policies keep out of it from the start.  FP32: 481,200 cells
// 14.0 us, 96^3 23.4, 1.54 million 37.8, 160^3 98.8, 256^3 462 (non-temporal
// 421); FP64: 64^3 14.2, 96^3 40.9, 128^3 102 (94), 160^3 231 (194).
inline double in_place_us(long long cells, bool f64, bool nt) {
    const double state = 19e-6 * (double)cells * (f64 ? 8 : 4);  // MB
    return nt ? 4.3 + 0.288 * state + 0.050 * std::max(0.0, state - 330.0)
              : 3.6 + 0.282 * state + 0.098 * std::max(0.0, state - 200.0);
}

// Equal walks of a launch: `groups` of them over nz planes, the wavefronts of
// beta and alpha of each, and the cells they step in all.
struct WalkSet {
    long long groups;
    int nz, waves;
    long long cells;
};

// The walks over domains in one launch.
struct WalkPlan {
    int threads = 0;
    std::vector<PairShape> shape;  // per domain
    std::vector<WalkSet> sets;
};
inline WalkPlan plan_walks(const std::vector<std::array<int, 3>> &dims, bool f64) {
    WalkPlan W;
    // The most work-items whose two LDS planes fit a compute unit (160 KB): the
    // larger the tile, the smaller its halo's share.  FP32 256^3 in tiles of
    // 1024 against 512: 336 and 343-375 us a step.
    W.threads = f64 ? 512 : 1024;
    std::vector<std::pair<long long, int>> planes;  // tiles per plane, planes
    for (const auto &d : dims) {
        W.shape.push_back(pair_shape(d[0], d[1], W.threads));
        planes.push_back({W.shape.back().tiles(), d[2]});
    }
    const int depth = dims.size() == 1 ? pair_depth(planes[0].second, planes[0].first, kPairSlots)
                                       : pair_depth_of_many(planes, kPairSlots);
    for (size_t i = 0; i < dims.size(); ++i) {
        const int Z = dims[i][2], chunks = (Z + depth - 1) / depth, nz = (Z + chunks - 1) / chunks;
        W.sets.push_back(WalkSet{planes[i].first * ((Z + nz - 1) / nz), nz,
                                 W.shape[i].beta_waves + W.shape[i].alpha_waves,
                                 (long long)dims[i][0] * dims[i][1] * Z});
    }
    return W;
}

// A pair by walks.  A plane takes a work-group its latency, however few columns
// it has, and a little more for every wavefront; kPairSlots run at once, in
// rounds, and the loads and stores take their share.  Measured / this, us a
// pair: FP32 96^3 34 / 38, 160^3 147 / 150, 256^3 655 / 677, 400x401x3 25 / 25,
// 1000x1000x3 148 / 136, 8x8x20000 189 / 174, 3000 of 8^3 266 / 259, 500 of
// 16^3 125 / 123; FP64 64^3 26 / 25, 128^3 199 / 180, 160^3 289 / 287,
// 300x300x3 37 / 38, 4000 of 8^3 428 / 410.  `filled`: where other streams'
// launches take the slots that are idle at its end.
inline double walks_us(const std::vector<WalkSet> &sets, bool f64, bool filled = false) {
    auto walk_us = [f64](const WalkSet &s) {
        return ((double)s.nz + 2.5) * (f64 ? 1.84 + 0.0385 * s.waves : 1.70 + 0.0167 * s.waves);
    };
    double sum = 0.0, longest = 0.0, shortest = 0.0;
    long long groups = 0, cells = 0;
    for (const WalkSet &s : sets) {
        const double t = walk_us(s);
        longest = std::max(longest, t);
        shortest = groups ? std::min(shortest, t) : t;
        sum += t * (double)s.groups;
        groups += s.groups;
        cells += s.cells;
    }
    double rounds = longest * (double)((groups + kPairSlots - 1) / kPairSlots);
    if (filled) {
        rounds = sum / (double)kPairSlots;
    } else if (shortest < longest) {  // each walk takes the slot that is free first
        if (groups > 64 * kPairSlots) {
            rounds = sum / (double)kPairSlots + 0.5 * longest;
        } else {
            std::priority_queue<double, std::vector<double>, std::greater<double>> free(
                std::greater<double>(), std::vector<double>((size_t)kPairSlots, 0.0));
            rounds = 0.0;
            for (const WalkSet &s : sets)
                for (long long k = 0; k < s.groups; ++k) {
                    const double end = free.top() + walk_us(s);
                    free.pop();
                    free.push(end);
                    rounds = std::max(rounds, end);
                }
        }
    }
    return (f64 ? 2.4 : 3.2) + rounds + (f64 ? 37.2e-6 : 20.4e-6) * (double)cells;
}

// The time to choose by.  A group's walks leave slots idle at their end, most of
// all where members differ, so that groups of several streams gain from pairs
// what one group on its own loses; as often the one as the other is assumed.  In
// place / pairs, us a half-step on its own and among others: 10 members of 17 to
// 58 cells an edge 17 / 21 and 12.5 / 10.9, 14 of 14 to 79 34 / 35 and 31 / 26.
inline double expected_walks_us(const std::vector<WalkSet> &sets, bool f64) {
    const double own = walks_us(sets, f64);
    return sets.size() > 1 ? 0.5 * (own + walks_us(sets, f64, true)) : own;
}

// Domains of fewer cells have too few columns to hide a walk's latency; us a
// step, in place / walks: FP32 64^3 8.7 / 10.3, 72^3 10.4 / 10.8, 80^3 14.3 /
// 13.2; FP64 48^3 7.7 / 10.0, 64^3 14.1 / 12.9.
constexpr long long walk_cells(bool f64) { return f64 ? 250000 : 480000; }

// Whether a sequence goes by walks.  They lose where a walk has few columns, or
// few planes for the two of its halo; in place / walks, us a half-step: FP32
// 3000 of 8^3 37.8 / 133, 500 of 16^3 47 / 63, 4x4x60000 25 / 275, 1000x1000x3
// 67 / 74; FP64 300x300x3 15.1 / 18.5, 400 of 12^3 33 / 51.  The margins keep
// the fit's error around equal times from costing more than 3 % on any of about
// 170 measured shapes and policies of one domain or equal members, each on its own.
// Of 24 batches of unequal members, 10 gain by pairs either way, 6 lose 2 to 4 % (one
// 16) on their own and gain 8 to 44 among others (one loses 2.5), 8 step in place.
inline bool walks_pay(const std::vector<WalkSet> &sets, bool f64, bool nt) {
    long long cells = 0;
    for (const WalkSet &s : sets) cells += s.cells;
    if (cells < walk_cells(f64)) return false;
    const double margin = f64 ? (nt ? 1.10 : 1.06) : (nt ? 1.07 : 1.045);
    return expected_walks_us(sets, f64) * margin <= 2.0 * in_place_us(cells, f64, nt);
}

// The same for domains that exchange faces (plan_faces): cells of the x faces
// and of the y and z faces, each from both sides.
struct FaceCells {
    long long x = 0, yz = 0;
};

// The pair takes five launches, or two with x faces only, and steps some cells
// again; the half-steps take their copies, or x faces in the step kernel, whose
// time varies more.  Below 335 MB, most of it in the last-level cache, either
// way can win by a quarter: us a half-step, in place / pairs, FP32 8 of 80^3
// with x faces in the kernel 140 / 117, copied 121 / 117, 125 of 32^3 148 /
// 162, 512 of 20^3 200 / 230; FP64 8 of 64^3 114 / 111, 4 of 150x150x20 98 /
// 121.  Above: FP32 8 of 128^3 480-570 / 374, 125 of 40^3 357 / 275, 100 of
// 16x16x200 221 / 280, 8 of 512x512x4 257 / 264; FP64 8 of 96^3 416-473 / 327,
// 8 of 300x300x4 339 / 370.  FP32 joined in x only with non-temporal accesses
// gains down to 84 MB (2 of 100^3 56-69 / 54, 3 of 40x100x100 42-52 / 40, with
// the default policy 52 / 54 and 38-44 / 40).  The FP64 non-temporal margin is the
// fit's error there; FP32 goes by equal times, since pairs lose less to other
// streams: 16 of 70^3 160 / 166 and, among others, 189 / 155, 12 of 92x70x65 177 /
// 146 and 188 / 136.
struct FaceTimes {
    double in_place, pairs;  // two half-steps
};
inline FaceTimes face_times(const std::vector<WalkSet> &sets, long long cells, const FaceCells &faces, bool f64, bool nt) {
    const double x = 1e-5 * (double)faces.x, yz = 1e-5 * (double)faces.yz;
    const double half = 2.0 * in_place_us(cells, f64, nt);
    return FaceTimes{f64 ? (nt ? 1.080 * half + 31.3 * x + 6.1 * yz : 1.127 * half + 25.1 * x + 5.6 * yz)
                         : (nt ? 1.155 * half + 20.4 * x + 2.4 * yz : 1.204 * half + 16.2 * x + 1.5 * yz),
                     f64 ? 3.0 + 1.19 * walks_us(sets, f64) + 35.7 * x + 9.5 * yz
                         : 15.7 + 1.23 * walks_us(sets, f64) + 25.8 * x + 4.7 * yz};
}
inline bool face_pairs_pay(const std::vector<WalkSet> &sets, const FaceCells &faces, bool f64, bool nt) {
    long long cells = 0;
    for (const WalkSet &s : sets) cells += s.cells;
    const double state = 19e-6 * (double)cells * (f64 ? 8 : 4);  // MB
    if (!f64 && nt && faces.yz == 0) return state >= 84.0;
    if (state < 335.0) return false;
    const FaceTimes t = face_times(sets, cells, faces, f64, nt);
    return t.pairs * (nt && f64 ? 1.065 : 1.0) <= t.in_place;
}

// What pairs gain on a half-step, us (at least a twentieth, where they pay at all).
inline double pairs_gain_us(const std::vector<WalkSet> &sets, const FaceCells *faces, bool f64, bool nt) {
    long long cells = 0;
    for (const WalkSet &s : sets) cells += s.cells;
    FaceTimes t{2.0 * in_place_us(cells, f64, nt), 0.0};
    if (faces) t = face_times(sets, cells, *faces, f64, nt);
    else t.pairs = expected_walks_us(sets, f64);
    return 0.5 * std::max(t.in_place - t.pairs, 0.05 * t.in_place);
}

// What the first pairs cost besides, us: the second buffers, tile tables and,
// of a group, its descriptors and the copies of its `comms`; an allocation takes
// about a microsecond a megabyte.  Of a solver, first run(4) in place / with
// that: 20^3 29 / 46-105, 96^3 110 / 240, 160^3 440 / 560; of a group, first
// step(4): 40 of 48^3 640 / 850-1200, 2x2x2 of 128^3 2350 / 2850-4800, 4x4x4 of
// 64^3 3400 / 6500.  `spare`: a destroyed solver's buffer is at hand.
inline double pairs_setup_us(double state_mb, bool group, size_t comms, bool spare) {
    return (spare ? (group ? 150.0 : 30.0) : (group ? 250.0 : 80.0) + state_mb) + 10.5 * (double)comms;
}

// Whether a sequence of `steps` half-steps is to pay that: once what it gains,
// with what `before` half-steps that went in place would have gained, makes up
// for it.  So short runs from new states stay as they were, and long ones and
// repeated ones lose at most that much again.
inline bool setup_repaid(double gain_us, double setup_us, long long before, long long steps) {
    return gain_us * (double)(before + steps) >= setup_us;
}

}  // namespace lbm
