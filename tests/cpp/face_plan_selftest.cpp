// Checks the plan by which members that exchange faces run as fused pairs: it
// is whole for the present members or empty, and its copies and rows cover
// every exchanged cell once.
#include <chrono>
#include <cstdio>

#include "face_plan.hpp"

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

typedef std::vector<std::array<int, 3>> Dims;

// both comms across the face between `low` and `high` along axis a
static void join(std::vector<GroupComm> &out, const Dims &d, int low, int high, int a) {
    for (int side = 0; side < 2; ++side) {
        const int m = side ? low : high, n = side ? high : low;  // the high member's low face first
        GroupComm c{m, n, {0, 0, 0}, {0, 0, 0}, {d[m][0], d[m][1], d[m][2]}, {0, 0, 0}};
        c.size[a] = 1;
        c.normal[a] = side ? -1 : 1;
        c.send_origin[a] = side ? d[m][a] - 2 : 1;
        c.recv_origin[a] = side ? d[m][a] - 1 : 0;
        out.push_back(c);
    }
}

static FacePlan plan(const Dims &d, const std::vector<GroupComm> &c, bool stops = false) {
    return plan_faces(d, stops, c, 4, [](const GroupComm &, int) { return 0x1fu; });
}

// What the launch tables read of a plan, for `members` members.
static void check_whole(const FacePlan &P, size_t members, const char *what) {
    CHECK(P.layers.size() == members, "%s: %zu layers, %zu members", what, P.layers.size(), members);
    if (!P.seams) {
        CHECK(P.seam_at.empty() && P.seam_nb.empty() && P.seam_bytes == 0, "%s: seams of nothing", what);
        return;
    }
    CHECK(P.seam_at.size() == 2 * members && P.seam_nb.size() == 2 * members, "%s: %zu of %zu", what, P.seam_at.size(),
          2 * members);
    for (size_t i = 0; i < P.seam_at.size(); ++i) {
        CHECK(P.seam_at[i] < P.seam_bytes, "%s: place %zu", what, P.seam_at[i]);
        CHECK(P.seam_nb[i] >= 0 && P.seam_nb[i] < (int)members, "%s: member %d", what, P.seam_nb[i]);
    }
}

static void check_empty(const FacePlan &P, const char *what) {
    CHECK(!P.pairs() && P.layers.empty() && !P.seams && P.seam_bytes == 0 && P.seam_at.empty() && P.seam_nb.empty() &&
              P.hops[0].empty() && P.hops[1].empty(),
          "%s: not empty", what);
}

int main() {
    Dims two{{20, 12, 10}, {20, 12, 10}};
    std::vector<GroupComm> x;
    join(x, two, 0, 1, 0);
    FacePlan P = plan(two, x);
    check_whole(P, 2, "two in x");
    CHECK(P.pairs() && P.seams && P.seam_bytes == 2u * 5 * 12 * 10 * 4 && P.hops[0].empty() && P.hops[1].empty(),
          "two in x: %zu bytes", P.seam_bytes);

    // the same group with a third member that stops, or is joined in no known way
    Dims three = two;
    three.push_back({9, 9, 9});
    P = plan(three, x, true);
    check_empty(P, "a member that stops");
    P = plan(three, x);
    check_whole(P, 3, "a member without faces");
    CHECK(P.layers[2] == 0, "faces %u", P.layers[2]);
    std::vector<GroupComm> odd = x;
    odd[0].size[1] = odd[1].size[1] = 7;
    check_empty(plan(two, odd), "part of a face");
    odd = x;
    odd.pop_back();
    check_empty(plan(two, odd), "no counterpart");
    Dims thin{{3, 12, 10}, {3, 12, 10}};
    std::vector<GroupComm> t;
    join(t, thin, 0, 1, 0);
    check_empty(plan(thin, t), "layers that overlap");
    odd = x;
    join(odd, two, 0, 1, 0);
    check_empty(plan(two, odd), "a face joined twice");

    // 2 x 2 x 2, and with unequal members, whose x faces are copied
    Dims eight(8, {14, 12, 10});
    for (int unequal = 0; unequal < 2; ++unequal) {
        if (unequal)
            for (int i = 1; i < 8; i += 2) eight[(size_t)i][0] = 15;
        std::vector<GroupComm> c;
        for (int i = 0; i < 8; ++i)
            for (int a = 0; a < 3; ++a)
                if (!(i >> a & 1)) join(c, eight, i, i | 1 << a, a);
        P = plan(eight, c);
        check_whole(P, 8, "eight");
        CHECK(P.seams == !unequal, "seams %d", (int)P.seams);
        for (int k = 0; k < 2; ++k)
            for (const HOp &h : P.hops[k]) {
                const std::array<int, 3> &d = eight[(size_t)h.dm];
                const SeamRows R(P.layers[(size_t)h.dm], d[1], d[2]);
                const int o[3] = {0, R.y0, R.z0}, sz[3] = {d[0], R.ny, R.nz};
                int io[3], is[3];
                if (P.seams) CHECK(!box_isect(h.dof, h.sz, o, sz, io, is), "a copy in the rows of pair_kernel");
                for (int a = 0; a < 3; ++a) CHECK(h.dof[a] >= 0 && h.dof[a] + h.sz[a] <= d[a], "copy outside");
            }
    }
    // many members: the plan's time grows with them, not with their square
    {
        const int n = 10;
        Dims many(n * n * n, {12, 12, 12});
        std::vector<GroupComm> c;
        for (int i = 0; i < n * n * n; ++i) {
            const int at[3] = {i % n, i / n % n, i / n / n}, step[3] = {1, n, n * n};
            for (int a = 0; a < 3; ++a)
                if (at[a] < n - 1) join(c, many, i, i + step[a], a);
        }
        const auto t0 = std::chrono::steady_clock::now();
        P = plan(many, c);
        const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        check_whole(P, many.size(), "a thousand");
        CHECK(s < 2.0, "a thousand members: %.1f s", s);
    }
    if (fails) {
        printf("%d failures\n", fails);
        return 1;
    }
    printf("face plan: ok\n");
    return 0;
}
