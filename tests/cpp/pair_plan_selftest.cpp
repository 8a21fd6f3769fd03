// Checks the tiles of the fused beta + alpha kernel against the indices the
// kernel forms from them: every cell is an inner column of exactly one tile,
// every gather lands in the domain, tiles that skip the linear wrap never
// leave it, and every neighbour alpha takes from LDS was computed.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "pair_plan.hpp"

using namespace lbm;

static int fails = 0;
#define CHECK(c, ...)                        \
    do {                                     \
        if (!(c)) {                          \
            if (++fails < 20) {              \
                printf("FAIL %s: ", #c);     \
                printf(__VA_ARGS__);         \
                printf("\n");                \
            }                                \
        }                                    \
    } while (0)

static long long wrap1(long long a, long long cells) {
    a = a < 0 ? a + cells : a;
    return a >= cells ? a - cells : a;
}

static void check(int X, int Y, int Z, int threads, int nz) {
    const PairShape s = pair_shape(X, Y, threads);
    std::vector<PairTile> tiles;
    pair_tiles(0, X, Y, Z, s, nz, tiles);
    const long long XY = (long long)X * Y, cells = XY * Z;
    std::vector<unsigned char> seen((size_t)cells, 0);
    CHECK(s.tiles() > 0 && s.beta_waves * 64 <= (threads + 63) / 64 * 64, "%dx%dx%d threads %d", X, Y, Z, threads);
    for (const PairTile &P : tiles) {
        const bool wrap = pair_wraps(P, X, (int)XY, (int)cells);
        const int pitch = pair_pitch(P, X);
        const long long last = P.org + (P.w == 0 ? P.h - 1 : P.w - 1 + (long long)X * (P.h - 1));
        std::vector<long long> at(threads, -1);  // LDS position -> in-plane position
        std::vector<char> held(threads, 0);
        long long columns = 0;
        for (int t = 0; t < threads; ++t) {
            const PairLane L = pair_beta_lane(P, X, t);
            if (L.pos < 0) continue;
            CHECK(L.pos < threads, "%dx%dx%d LDS position %d of %d", X, Y, Z, L.pos, threads);
            if (L.pos >= threads) continue;
            CHECK(!held[L.pos], "two lanes hold position %d", L.pos);
            held[L.pos] = 1;
            at[L.pos] = L.p;
            ++columns;
            CHECK(L.p >= P.org && L.p <= last, "column outside the tile");
            for (int z = P.z0 - 1; z <= P.z0 + P.nz; ++z)
                for (int dz = -1; dz <= 1; ++dz)
                    for (int dy = -1; dy <= 1; ++dy)
                        for (int dx = -1; dx <= 1; ++dx) {
                            const long long g = L.p + XY * (z + dz) + X * dy + dx;
                            const long long w = wrap ? wrap1(g, cells) : g;
                            CHECK(w >= 0 && w < cells, "%dx%dx%d gather %lld (wrap %d)", X, Y, Z, g, (int)wrap);
                        }
        }
        CHECK(columns == (P.w == 0 ? P.h : (long long)P.w * P.h), "%dx%dx%d threads %d: %lld columns", X, Y, Z, threads, columns);
        for (int t = 0; t < threads; ++t) {
            const PairLane L = pair_alpha_lane(P, X, t);
            if (L.pos < 0) continue;
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    const int q = L.pos - (dx + pitch * dy);
                    CHECK(q >= 0 && q < threads && held[q], "%dx%dx%d LDS neighbour %d", X, Y, Z, q);
                    if (q >= 0 && q < threads && held[q])
                        CHECK(at[q] == L.p - dx - (long long)X * dy, "LDS neighbour is another column");
                }
            for (int z = P.z0; z < P.z0 + P.nz; ++z) {
                const long long g = L.p + XY * z;
                CHECK(g >= 0 && g < cells, "store %lld", g);
                if (g >= 0 && g < cells) seen[(size_t)g]++;
            }
        }
    }
    for (long long g = 0; g < cells; ++g) CHECK(seen[(size_t)g] == 1, "%dx%dx%d cell %lld stored %d times", X, Y, Z, g, seen[(size_t)g]);
}

// the boxes of the small-domain kernel
static void check_box(int X, int Y, int Z, int held, int threads, int resident) {
    const BoxShape b = box_shape(X, Y, Z, held, threads, resident, 256);
    CHECK(b.cost > 0, "%dx%dx%d: no boxes", X, Y, Z);
    if (b.cost <= 0) return;
    std::vector<PairTile> tiles;
    box_tiles(0, X, Y, Z, b, tiles);
    const long long XY = (long long)X * Y, cells = XY * Z;
    std::vector<unsigned char> seen((size_t)cells, 0);
    for (const PairTile &P : tiles) {
        const bool wrap = pair_wraps(P, X, (int)XY, (int)cells);
        const int w = P.w, wh = P.w * P.h, n = wh * (P.nz + 2);
        CHECK(n <= held, "%dx%dx%d box of %d cells, %d held", X, Y, Z, n, held);
        auto cell = [&](int e) {
            const int tz = e / wh, r = e - tz * wh, ty = r / w;
            return P.org + r - ty * w + (long long)X * ty + XY * (P.z0 - 1 + tz);
        };
        for (int e = 0; e < n; ++e)
            for (int dz = -1; dz <= 1; ++dz)
                for (int dy = -1; dy <= 1; ++dy)
                    for (int dx = -1; dx <= 1; ++dx) {
                        const long long g = cell(e) + XY * dz + X * dy + dx, v = wrap ? wrap1(g, cells) : g;
                        CHECK(v >= 0 && v < cells, "%dx%dx%d box gather %lld (wrap %d)", X, Y, Z, g, (int)wrap);
                    }
        const int iw = P.w - 2, iwh = iw * (P.h - 2);
        for (int e = 0; e < iwh * P.nz; ++e) {
            const int tz = e / iwh, r = e - tz * iwh, ty = r / iw, tx = r - ty * iw;
            const int pos = (tz + 1) * wh + (ty + 1) * w + tx + 1;
            const long long g = P.org + tx + 1 + (long long)X * (ty + 1) + XY * (P.z0 + tz);
            CHECK(pos - (1 + w + wh) >= 0 && pos + 1 + w + wh < n, "box neighbour out of LDS");
            CHECK(cell(pos) == g && g >= 0 && g < cells, "box store %lld", g);
            if (g >= 0 && g < cells) seen[(size_t)g]++;
        }
    }
    for (long long g = 0; g < cells; ++g) CHECK(seen[(size_t)g] == 1, "%dx%dx%d box cell %lld stored %d times", X, Y, Z, g, seen[(size_t)g]);
}

int main() {
    srand(7);
    for (int threads : {256, 512, 1024})
        for (int k = 0; k < 60; ++k) {
            const int X = 3 + rand() % (k % 3 ? 40 : 300), Y = 3 + rand() % (k % 4 ? 40 : 90), Z = 3 + rand() % 12;
            check(X, Y, Z, threads, 1 + rand() % Z);
        }
    for (int threads : {256, 512, 1024})
        for (int X : {3, 4, 24, 32, 64, 97, 128, 150, 254, 255, 256, 300, 510, 512, 1022})
            for (int Y : {3, 16, 33}) check(X, Y, 3, threads, 2);
    for (int Z = 3; Z < 200; ++Z)
        for (long long tiles : {1ll, 7ll, 90ll, 2000ll}) {
            const int nz = pair_depth(Z, tiles, 512);
            CHECK(nz >= 1 && nz <= Z, "depth %d of %d", nz, Z);
        }
    for (int held : {704, 1056, 2048})
        for (int k = 0; k < 40; ++k)
            check_box(3 + rand() % (k % 4 ? 40 : 200), 3 + rand() % (k % 5 ? 40 : 150), 3 + rand() % (k % 3 ? 30 : 100), held,
                      held == 704 ? 704 : held / 2, 1 + k % 2);
    for (int held : {704, 1056, 2048}) {
        check_box(3, 3, 3, held, 512, 1);
        check_box(500, 3, 3, held, 512, 1);
        check_box(3, 500, 3, held, 512, 1);
        check_box(3, 3, 900, held, 512, 1);
        check_box(64, 64, 64, held, 512, 1);
    }
    if (fails) {
        printf("%d failures\n", fails);
        return 1;
    }
    printf("pair plan: ok\n");
    return 0;
}
