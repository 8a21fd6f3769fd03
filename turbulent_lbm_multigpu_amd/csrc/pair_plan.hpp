// pair_plan.hpp -- tiles of the fused beta + alpha kernel (pair_kernel).
// Plain C++: the plan is checked on the CPU.
#pragma once

#include <algorithm>
#include <utility>
#include <vector>

namespace lbm {

#if defined(__HIPCC__)
#define LBM_PAIR_FN __host__ __device__ __forceinline__
#else
#define LBM_PAIR_FN inline
#endif

// One work-group of the pair kernel: `nz` planes from z0 of a tile in x-y,
// halo columns included: w x h columns, or, with w == 0, a run of h
// consecutive positions of rows of X.  `org` is the in-plane linear position
// of the first column; it may be negative and columns may lie past the plane:
// positions are linear and wrap at the ends of the domain, as the streaming
// does.
struct PairTile {
    int dom;
    int org;
    int z0, nz;
    int w, h;
};

// A column of a work-item: its LDS position in the tile (-1: none) and its
// in-plane linear position.
struct PairLane {
    int pos, p;
};

// LDS positions of one row of a tile
LBM_PAIR_FN int pair_pitch(const PairTile &P, int X) { return P.w ? P.w : X; }

// The column whose beta work-item t computes: the tile's columns row by row.
LBM_PAIR_FN PairLane pair_beta_lane(const PairTile &P, int X, int t) {
    if (P.w == 0) return PairLane{t < P.h ? t : -1, P.org + t};
    const int ty = t / P.w;
    return PairLane{ty < P.h ? t : -1, P.org + t - ty * P.w + X * ty};
}

// The inner column whose alpha work-item t computes.
LBM_PAIR_FN PairLane pair_alpha_lane(const PairTile &P, int X, int t) {
    if (P.w == 0) return PairLane{t < P.h - 2 * (X + 1) ? t + X + 1 : -1, P.org + t + X + 1};
    const int iw = P.w - 2, ty = t / iw, tx = t - ty * iw;
    return PairLane{ty < P.h - 2 ? (ty + 1) * P.w + tx + 1 : -1, P.org + tx + 1 + X * (ty + 1)};
}

// Whether a gather of the tile leaves the domain and wraps: those of planes
// z0-1 .. z0+nz reach planes z0-2 .. z0+nz+1.
LBM_PAIR_FN bool pair_wraps(const PairTile &P, int X, int XY, int cells) {
    const int last = P.org + (P.w == 0 ? P.h - 1 : P.w - 1 + X * (P.h - 1));
    return P.org - 1 - X + XY * (P.z0 - 2) < 0 || last + 1 + X + XY * (P.z0 + P.nz + 1) >= cells;
}

// A domain that exchanges faces: bit 2a (2a + 1) of `layers` is set where the
// low (high) end of axis a has a neighbour.  Whether coordinate c of that axis
// (extent n) is in the ghost layer there or in the layer next to it.
LBM_PAIR_FN bool in_layers(unsigned layers, int a, int c, int n) {
    return ((layers >> (2 * a) & 1u) != 0 && c < 2) || ((layers >> (2 * a + 1) & 1u) != 0 && c >= n - 2);
}

// The rows (y, z) of a domain that are in no layer of y or z, by y, then z: in
// those pair_kernel exchanges x faces itself.  What comes in over a face are
// the kSeamPops populations that beta moves over it, by population (in their
// order) and row.
constexpr int kSeamPops = 5;
struct SeamRows {
    int y0, z0, ny, nz;
    LBM_PAIR_FN SeamRows(unsigned layers, int Y, int Z)
        : y0(layers >> 2 & 1u ? 2 : 0), z0(layers >> 4 & 1u ? 2 : 0), ny(Y - y0 - (layers >> 3 & 1u ? 2 : 0)),
          nz(Z - z0 - (layers >> 5 & 1u ? 2 : 0)) {}
    LBM_PAIR_FN int count() const { return ny * nz; }
    LBM_PAIR_FN bool has(int y, int z) const { return y >= y0 && y < y0 + ny && z >= z0 && z < z0 + nz; }
};

// An x face of domain `dom`, beyond it `nb`, as a range of blocks of
// seam_beta_kernel.
struct SeamFace {
    int dom, side, nb;
    int block_begin;
};

// Planes of a domain at an exchanged face, a range of blocks of
// layer_alpha_kernel.
struct LayerBox {
    int dom, axis;
    int o[3], s[3];
    int block_begin;
};

// The boxes of a domain, those of x faces unless `seams`; a cell of several
// belongs to the one of the last axis.
inline void layer_boxes(int dom, unsigned layers, const int *dims, bool seams, std::vector<LayerBox> &out) {
    for (int a = seams ? 1 : 0; a < 3; ++a)
        for (int side = 0; side < 2; ++side) {
            if (!(layers >> (2 * a + side) & 1u)) continue;
            LayerBox b{dom, a, {0, 0, 0}, {dims[0], dims[1], dims[2]}, 0};
            b.o[a] = side ? dims[a] - 2 : 0;
            b.s[a] = 2;
            out.push_back(b);
        }
}

// How a pair launch is made.
struct PairLaunch {
    int threads = 0;
    bool layers = false;  // the domains exchange faces between beta and alpha (DomDev::layers)
    int box_cells = 0;  // > 0: tiles are boxes of at most this many columns x planes (pair_box_kernel)
    int xcd_map = 0;  // see step_kernel
};

// Shape of a domain's tiles in x-y for work-groups of `threads`.
struct PairShape {
    bool run = false;  // runs of consecutive positions (pitch X); else rectangles
    int tx = 0, ty = 0;  // inner columns per tile: tx positions (run), or tx by ty
    int nx = 0, ny = 0;  // tiles per plane: nx (run), or nx by ny
    int tiles() const { return run ? nx : nx * ny; }
    int beta_waves = 0, alpha_waves = 0;  // of a full tile
};

// A tile computes beta on its inner columns and a halo of one column around
// them, so the halo is work done twice (and read twice).  Of all tiles that
// fit the work-group, the fewest wavefronts of beta and alpha per plane, with
// a price on narrow rows, whose lines are fetched for single columns at their
// ends: whole rows as runs of consecutive positions (halo X + 1 positions on
// each side) suit short rows, rectangles long ones.  FP32 256^3, rows of 32,
// 64 and 128 inner columns: 367, 342 and 315-330 us a step.
inline PairShape pair_shape(int X, int Y, int threads) {
    PairShape best;
    double best_cost = -1;
    auto take = [&](PairShape s, int inner, int all) {
        s.alpha_waves = (inner + 63) / 64;
        s.beta_waves = (all + 63) / 64;
        if (all > threads || inner < 1) return;
        const double cost = (double)s.tiles() * (s.beta_waves + s.alpha_waves) * (s.run ? 1.0 : 1.0 + 25.0 / s.tx);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = s;
        }
    };
    const long long XY = (long long)X * Y;
    const int len = threads - 2 * (X + 1);
    if (len >= 1) {
        PairShape s;
        s.run = true;
        s.nx = (int)((XY + len - 1) / len);
        s.tx = (int)((XY + s.nx - 1) / s.nx);
        s.ny = 1;
        take(s, s.tx, s.tx + 2 * (X + 1));
    }
    for (int n = 1; n <= X; ++n) {
        const int tx = (X + n - 1) / n;
        if (tx < 6 && n > 1) break;
        PairShape s;
        s.nx = (X + tx - 1) / tx;
        s.tx = tx;
        const int rows = threads / (tx + 2) - 2;  // the most that fit, evened out over the plane
        if (rows < 1) continue;
        s.ny = (Y + rows - 1) / rows;
        s.ty = (Y + s.ny - 1) / s.ny;
        take(s, s.tx * s.ty, (s.tx + 2) * (s.ty + 2));
    }
    return best;
}

// Planes per work-group: a work-group walks nz + 2 planes (the two at its
// ends are halo), so long walks waste least, but `slots` work-groups run at
// once and the last round of them should be full.
inline int pair_depth(int Z, long long tiles_per_plane, long long slots) {
    int best = Z;
    double best_cost = -1.0;
    for (int n = 1; n <= Z; ++n) {  // chunks along z
        const int nz = (Z + n - 1) / n;
        if (n > 1 && (Z + nz - 1) / nz != n) continue;
        const long long blocks = tiles_per_plane * n;
        const long long rounds = (blocks + slots - 1) / slots;
        const double cost = (double)rounds * (nz + 2.0 + 0.5);
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best = nz;
        }
        if (nz == 1) break;
    }
    return best;
}

// The same for many domains in one launch ((tiles per plane, planes) each):
// the walks are of all lengths and fill the device one after another, so
// only their number and the length of the last ones matter.
inline int pair_depth_of_many(const std::vector<std::pair<long long, int>> &planes, long long slots) {
    int best = 1;
    double best_cost = -1.0;
    for (int nz : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128}) {
        double work = 0.0;
        for (const auto &p : planes) work += (double)p.first * (p.second + 2.5 * ((p.second + nz - 1) / nz));
        const double cost = work / (double)slots + 0.7 * (nz + 2.5);
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best = nz;
        }
    }
    return best;
}

// Appends the tiles of domain `dom`, x fastest, then y, then z chunks.
inline void pair_tiles(int dom, int X, int Y, int Z, const PairShape &s, int nz, std::vector<PairTile> &out) {
    const int XY = X * Y;
    for (int z0 = 0; z0 < Z; z0 += nz) {
        const int dz = std::min(nz, Z - z0);
        if (s.run) {
            for (int i = 0; i < s.nx; ++i) {
                const int p0 = i * s.tx, len = std::min(s.tx, XY - p0);
                if (len <= 0) break;
                out.push_back(PairTile{dom, p0 - X - 1, z0, dz, 0, len + 2 * (X + 1)});
            }
            continue;
        }
        for (int j = 0; j < s.ny; ++j) {
            const int y0 = j * s.ty, ty = std::min(s.ty, Y - y0);
            if (ty <= 0) break;
            for (int i = 0; i < s.nx; ++i) {
                const int x0 = i * s.tx, tx = std::min(s.tx, X - x0);
                if (tx <= 0) break;
                out.push_back(PairTile{dom, x0 - 1 + X * (y0 - 1), z0, dz, tx + 2, ty + 2});
            }
        }
    }
}

// Boxes of the small-domain pair kernel: a work-group holds the beta values of
// a whole box, halo included, in LDS.  `cells`: what its LDS holds, `threads`
// its work-items, `resident` how many of it a compute unit runs at once.
struct BoxShape {
    int bx = 0, by = 0, bz = 0;  // inner cells per box and axis
    double cost = -1.0;
};

// Small domains leave compute units idle or repeat much of beta on the halo;
// this picks the boxes whose rounds of work-groups take least: the wavefronts
// of beta and alpha that share a compute unit, plus a load latency for each
// pass over the box.  Units: a wavefront's collision.
inline BoxShape box_shape(int X, int Y, int Z, int cells, int threads, int resident, long long units) {
    // even splits of an axis into boxes of at least `least` cells, at most 32
    auto splits = [](int n, int least) {
        std::vector<int> v;
        for (int k = 1; k <= n; ++k) {
            const int b = (n + k - 1) / k;
            if (b < least && k > 1) break;
            if (b <= 32 && (v.empty() || v.back() != b)) v.push_back(b);
        }
        return v;
    };
    const std::vector<int> sx = splits(X, 6), sy = splits(Y, 4), sz = splits(Z, 1);
    BoxShape best;
    for (int bx : sx)
        for (int by : sy)
            for (int bz : sz) {
                const int ext = (bx + 2) * (by + 2) * (bz + 2);
                if (ext > cells) continue;
                const int in = bx * by * bz;
                const long long blocks = (long long)((X + bx - 1) / bx) * ((Y + by - 1) / by) * ((Z + bz - 1) / bz);
                const long long per = (blocks + units - 1) / units;  // work-groups a compute unit runs in all
                const long long rounds = (per + resident - 1) / resident;
                const double waves = (double)((ext + 63) / 64 + (in + 63) / 64);
                const double passes = (double)((ext + threads - 1) / threads + (in + threads - 1) / threads);
                const double cost = (double)per * waves + (double)rounds * 6.0 * passes;
                if (best.cost < 0.0 || cost < best.cost) best = BoxShape{bx, by, bz, cost};
            }
    return best;
}

inline void box_tiles(int dom, int X, int Y, int Z, const BoxShape &b, std::vector<PairTile> &out) {
    for (int z0 = 0; z0 < Z; z0 += b.bz)
        for (int y0 = 0; y0 < Y; y0 += b.by)
            for (int x0 = 0; x0 < X; x0 += b.bx)
                out.push_back(PairTile{dom, x0 - 1 + X * (y0 - 1), z0, std::min(b.bz, Z - z0),
                                       std::min(b.bx, X - x0) + 2, std::min(b.by, Y - y0) + 2});
}

}  // namespace lbm
