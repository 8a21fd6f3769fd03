// Checks the choice between fused pairs and half-steps in place against shapes
// that were measured both ways: the faster way where they differ by more than
// the fit's error.
#include <cmath>
#include <cstdio>

#include "pair_cost.hpp"

using namespace lbm;

// us a half-step in place and by pairs, `n` domains of x * y * z
struct Measured {
    int n, x, y, z;
    double in_place, pairs;
};

static const Measured F32[] = {
    {1, 400, 401, 3, 14.0, 12.7},    {1, 300, 300, 6, 16.1, 14.0},    {1, 12, 200, 210, 14.7, 13.4},
    {1, 500, 4, 250, 13.9, 11.4},    {1, 83, 79, 77, 14.8, 14.2},     {1, 90, 90, 90, 20.5, 16.1},
    {1, 96, 96, 96, 23.4, 17.1},     {1, 128, 128, 128, 48.8, 39.4},  {1, 160, 160, 160, 98.8, 73.8},
    {1, 256, 256, 256, 462, 327},    {1, 2000, 1500, 3, 248, 203},    {1, 3, 1000, 1000, 68.3, 55.7},
    {1, 30, 30, 1200, 27.3, 20.3},   {1, 1000, 1000, 3, 66.6, 74.0},  {1, 16, 16, 8000, 48.2, 53.8},
    {1, 8, 8, 20000, 32.1, 94.5},    {1, 4, 4, 60000, 24.8, 274},     {1, 257, 130, 15, 13.9, 14.6},
    {118, 16, 16, 16, 14.1, 18.4},   {500, 16, 16, 16, 47.0, 62.6},   {300, 12, 12, 12, 14.9, 32.8},
    {3000, 8, 8, 8, 37.8, 133},      {40, 3, 50, 100, 17.9, 29.1},    {40, 100, 50, 3, 17.1, 18.7},
    {400, 8, 8, 64, 38.9, 148},      {200, 20, 20, 20, 38.5, 43.1},   {3000, 12, 12, 12, 148, 229},
    {5, 48, 48, 48, 17.0, 13.7},     {16, 48, 48, 48, 41.8, 35.6},    {600, 24, 24, 24, 231, 149},
    {400, 100, 50, 3, 169, 127},     {40, 64, 64, 64, 285, 205},        {1, 512, 512, 6, 37.7, 32.2},
};
static const Measured F64[] = {
    {1, 64, 64, 64, 14.2, 13.0},     {1, 68, 68, 68, 17.1, 14.6},     {1, 80, 80, 80, 25.1, 20.2},
    {1, 96, 96, 96, 40.9, 32.2},     {1, 160, 160, 160, 231, 145},    {1, 16, 16, 4000, 46.6, 39.6},
    {1, 3, 700, 700, 64.9, 50.7},    {1, 700, 700, 5, 119, 105},      {1, 300, 300, 3, 15.1, 18.5},
    {1, 520, 33, 17, 15.9, 17.5},    {1, 500, 500, 4, 46.0, 50.5},    {1, 8, 8, 10000, 30.9, 55.6},
    {1, 130, 130, 20, 18.6, 19.1},   {600, 8, 8, 8, 16.9, 37.3},      {400, 12, 12, 12, 33.5, 50.6},
    {80, 16, 16, 16, 18.4, 21.8},    {20, 100, 50, 3, 16.5, 18.6},    {4000, 8, 8, 8, 98.5, 214},
    {2000, 16, 16, 16, 447, 284},    {20, 64, 64, 64, 288, 186},      {40, 20, 20, 20, 18.6, 15.3},
    {200, 100, 50, 3, 170, 142},     {8, 48, 48, 48, 40.7, 36.5},
};
// with non-temporal accesses in place
static const Measured NT32[] = {
    {1, 256, 256, 256, 421, 327}, {500, 16, 16, 16, 49.8, 62.7}, {2000, 16, 16, 16, 195, 212}, {1, 96, 96, 96, 23.5, 17.1},
};
static const Measured NT64[] = {
    {1, 128, 128, 128, 94.5, 99.6}, {1, 1000, 1000, 3, 141, 145}, {1, 160, 160, 160, 194, 145}, {1, 80, 80, 80, 26.6, 20.1},
};

// Members nx * ny * nz of x * y * z that exchange all their faces.
struct Joined {
    int n[3];
    int d[3];
    bool f64, nt, pairs;
};
static const Joined FACES[] = {
    {{2, 2, 2}, {128, 128, 128}, false, false, true},  // 480-570 / 374
    {{2, 2, 2}, {128, 128, 128}, false, true, true},   // 421-496 / 374
    {{5, 5, 5}, {40, 40, 40}, false, false, true},     // 357 / 275
    {{2, 2, 2}, {300, 300, 10}, false, false, true},   // 222-249 / 195
    {{2, 2, 2}, {88, 88, 88}, false, false, true},     // 184 / 143
    {{2, 1, 1}, {160, 160, 160}, false, false, true},  // 277 / 175
    {{10, 10, 1}, {16, 16, 200}, false, false, false}, // 221 / 280
    {{1, 1, 8}, {512, 512, 4}, false, false, false},   // 257 / 264
    {{4, 1, 4}, {70, 70, 70}, false, true, true},      // 160 / 166, among others 189 / 155
    {{2, 3, 2}, {92, 70, 65}, false, true, true},      // 177 / 146, among others 188 / 136
    {{5, 5, 5}, {32, 32, 32}, false, false, false},    // 148 / 162
    {{8, 8, 8}, {20, 20, 20}, false, false, false},    // 200 / 230
    {{2, 2, 2}, {12, 200, 200}, false, false, false},  // 118-122 / 127
    {{2, 1, 1}, {60, 140, 140}, false, false, false},  // 57 / 62
    {{2, 1, 1}, {60, 140, 140}, false, true, true},    // 67-73 / 61
    {{3, 1, 1}, {40, 100, 100}, false, true, true},    // 42-52 / 40
    {{2, 2, 2}, {80, 80, 80}, true, false, true},      // 257-279 / 183
    {{2, 2, 2}, {96, 96, 96}, true, true, true},       // 364-398 / 327
    {{4, 4, 4}, {40, 40, 40}, true, false, true},      // 284-315 / 236
    {{2, 2, 2}, {300, 300, 4}, true, false, false},    // 339 / 370
    {{2, 2, 2}, {150, 150, 10}, true, false, false},   // 101-121 / 131
    {{4, 4, 4}, {32, 32, 32}, true, false, false},     // 114 / 135
};

static int fails = 0;

template <size_t N>
static void check(const Measured (&table)[N], bool f64, bool nt) {
    for (const Measured &m : table) {
        const std::vector<std::array<int, 3>> dims((size_t)m.n, {m.x, m.y, m.z});
        const WalkPlan W = plan_walks(dims, f64);
        const long long cells = (long long)m.n * m.x * m.y * m.z;
        const double in_place = in_place_us(cells, f64, nt), walks = walks_us(W.sets, f64) / 2;
        const bool want = m.pairs < m.in_place, got = walks_pay(W.sets, f64, nt);
        // both fits within a fifth, and the faster way taken
        const bool fit = in_place > 0.8 * m.in_place && in_place < 1.2 * m.in_place && walks > 0.78 * m.pairs && walks < 1.25 * m.pairs;
        if (want == got && fit) continue;
        ++fails;
        printf("FAIL: %d of %dx%dx%d f%d nt %d: in place %.1f (measured %.1f), pairs %.1f (%.1f), pairs taken %d\n", m.n,
               m.x, m.y, m.z, f64 ? 64 : 32, (int)nt, in_place, m.in_place, walks, m.pairs, (int)got);
    }
}

static void check_faces() {
    for (const Joined &m : FACES) {
        const std::vector<std::array<int, 3>> dims((size_t)(m.n[0] * m.n[1] * m.n[2]), {m.d[0], m.d[1], m.d[2]});
        FaceCells f;
        f.x = 2ll * (m.n[0] - 1) * m.n[1] * m.n[2] * m.d[1] * m.d[2];
        f.yz = 2ll * (m.n[1] - 1) * m.n[0] * m.n[2] * m.d[0] * m.d[2] +
               2ll * (m.n[2] - 1) * m.n[0] * m.n[1] * m.d[0] * m.d[1];
        const WalkPlan W = plan_walks(dims, m.f64);
        if ((walks_pay(W.sets, m.f64, m.nt) && face_pairs_pay(W.sets, f, m.f64, m.nt)) == m.pairs) continue;
        ++fails;
        printf("FAIL: %dx%dx%d of %dx%dx%d f%d nt %d: pairs are to be taken: %d\n", m.n[0], m.n[1], m.n[2], m.d[0],
               m.d[1], m.d[2], m.f64 ? 64 : 32, (int)m.nt, (int)m.pairs);
    }
}

int main() {
    check_faces();
    check(F32, false, false);
    check(F64, true, false);
    check(NT32, false, true);
    check(NT64, true, true);
    if (!walks_pay(plan_walks({{{96, 96, 96}}}, false).sets, false, false) ||
        walks_pay(plan_walks({{{72, 72, 72}}}, false).sets, false, false)) {
        ++fails;
        printf("FAIL: the least cells\n");
    }
    // the second buffer: not for a first short run, but for a long one or for many
    {
        const std::vector<WalkSet> sets = plan_walks({{{96, 96, 96}}}, false).sets;
        const double gain = pairs_gain_us(sets, nullptr, false, false), setup = pairs_setup_us(67.2, false, 0, false);
        if (setup_repaid(gain, setup, 0, 4) || !setup_repaid(gain, setup, 0, 200) || !setup_repaid(gain, setup, 196, 4) ||
            pairs_setup_us(67.2, true, 24, false) <= setup) {
            ++fails;
            printf("FAIL: gain %.1f a half-step, setup %.1f\n", gain, setup);
        }
        // with a buffer at hand the size does not count: a first run of 12 has them at once
        const double at_hand = pairs_setup_us(67.2, false, 0, true);
        if (setup_repaid(gain, setup, 0, 12) || !setup_repaid(gain, at_hand, 0, 12) || at_hand >= setup ||
            at_hand != pairs_setup_us(1000, false, 0, true) || pairs_setup_us(67.2, true, 24, true) <= at_hand) {
            ++fails;
            printf("FAIL: gain %.1f a half-step, setup %.1f and with a spare %.1f\n", gain, setup, at_hand);
        }
    }
    // idle slots at a launch's end count half: nearly equal lengths that fill
    // them, and one round and a bit of unequal ones
    {
        const std::vector<WalkSet> even = plan_walks(std::vector<std::array<int, 3>>(200, {24, 24, 24}), false).sets;
        std::vector<std::array<int, 3>> few;
        for (int n = 17; n <= 58; n += 4) few.push_back({n, 60 - n / 2, n});
        const std::vector<WalkSet> ragged = plan_walks(few, false).sets;
        for (const auto &sets : {even, ragged}) {
            const double own = walks_us(sets, false), filled = walks_us(sets, false, true), e = expected_walks_us(sets, false);
            if (filled <= own + 1e-9 && std::abs(e - 0.5 * (own + filled)) < 1e-9) continue;
            ++fails;
            printf("FAIL: own %.1f, filled %.1f, expected %.1f\n", own, filled, e);
        }
        const std::vector<WalkSet> one = plan_walks({{{100, 100, 100}}}, false).sets;
        if (expected_walks_us(one, false) != walks_us(one, false)) ++fails, printf("FAIL: a domain on its own\n");
    }
    // unequal members: the long ones decide how the last slots empty
    std::vector<std::array<int, 3>> mixed(40, {64, 64, 64});
    mixed.resize(60, {24, 24, 24});
    if (!walks_pay(plan_walks(mixed, false).sets, false, false)) {
        ++fails;
        printf("FAIL: unequal members\n");
    }
    if (fails) {
        printf("%d failures\n", fails);
        return 1;
    }
    printf("pair cost: ok\n");
    return 0;
}
