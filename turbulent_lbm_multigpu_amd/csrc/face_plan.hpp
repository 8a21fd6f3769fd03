// face_plan.hpp -- how members that exchange faces run as fused pairs
// (pair_kernel).  Plain C++: the plan is checked on the CPU.
#pragma once

#include <stddef.h>

#include <map>

#include "exchange_plan.hpp"
#include "pair_plan.hpp"

namespace lbm {

// A comm of a group: `member` receives across a face from `dst`.
struct GroupComm {
    int member, dst;
    int send_origin[3], recv_origin[3], size[3], normal[3];
};

// The counterparts of comms: the partner's comm across the same face (its first).
class Partners {
  public:
    explicit Partners(const std::vector<GroupComm> &comms) {
        for (const GroupComm &c : comms) at_.insert({key(c.member, c.dst, c.normal, 1), &c});
    }
    const GroupComm *of(const GroupComm &c) const {
        const auto it = at_.find(key(c.dst, c.member, c.normal, -1));
        return it == at_.end() ? nullptr : it->second;
    }

  private:
    typedef std::array<int, 5> Key;
    static Key key(int member, int dst, const int *n, int sign) {
        return Key{{member, dst, sign * n[0], sign * n[1], sign * n[2]}};
    }
    std::map<Key, const GroupComm *> at_;
};

// The two copies of a comm and its counterpart: [0] after alpha, [1] after
// beta, with the populations each of them takes.
inline void comm_copies(const GroupComm &c, const GroupComm &p, uint32_t alpha_mask, uint32_t beta_mask, HOp *h) {
    h[0] = HOp{c.dst, c.member, {}, {}, {}, alpha_mask};
    // after beta: neighbour's ghost layer -> my inner layer, n.e > 0 only (src/CController.hpp:322-383)
    h[1] = HOp{c.dst, c.member, {}, {}, {}, beta_mask};
    for (int ax = 0; ax < 3; ++ax) {
        h[0].so[ax] = p.send_origin[ax];
        h[0].dof[ax] = c.recv_origin[ax];
        h[1].so[ax] = p.recv_origin[ax];
        h[1].dof[ax] = c.send_origin[ax];
        h[0].sz[ax] = h[1].sz[ax] = c.size[ax];
    }
}

// Empty (no layers, no seams) where the members do not run as pairs.
struct FacePlan {
    std::vector<unsigned> layers;  // per member, the faces (DomDev::layers)
    std::vector<HOp> hops[2];      // the copies after alpha ([0]) and beta ([1])
    bool seams = false;            // x faces inside pair_kernel (SeamRows), with
    size_t seam_bytes = 0;         // what comes in over them, all members',
    std::vector<size_t> seam_at;   // per member and side, where its part starts
    std::vector<int> seam_nb;      // and the member beyond
    bool pairs() const { return !layers.empty(); }
};

// Whether members that exchange faces can run as fused pairs: every comm joins
// a whole face, ghost layer and the one next to it, with its counterpart, no
// member stops, and the copies of the three axes resolve to one set.  In such
// a pair the cells of the layers, whose alpha needs the exchange after beta,
// keep beta's values in the new buffer; there follow the copies after beta,
// alpha of the layers (layer_alpha_kernel) and the copies after alpha.  x faces
// are pair_kernel's own (SeamRows).  256^3 FP32 in 2x2x2: pair_kernel 620 us,
// before it seam_beta_kernel 89, after it 12 + 13 + 9, where beta, alpha and
// two copies in place took 858.  `masks(c, k)`: the populations of comm_copies.
template <class Masks>
FacePlan plan_faces(const std::vector<std::array<int, 3>> &dims, bool stops, const std::vector<GroupComm> &comms,
                    size_t elem, Masks &&masks) {
    if (stops || dims.empty()) return FacePlan{};
    FacePlan P;
    P.layers.assign(dims.size(), 0u);
    std::vector<HOp> phase[2][3];
    const Partners partners(comms);
    for (const GroupComm &c : comms) {
        const GroupComm *p = partners.of(c);
        if (!p) return FacePlan{};
        const int a = c.normal[0] ? 0 : c.normal[1] ? 1 : 2, side = c.normal[a] == 1 ? 0 : 1;
        for (const GroupComm *q : {&c, p}) {
            const std::array<int, 3> &d = dims[(size_t)q->member];
            const bool low = q->normal[a] == 1;
            for (int ax = 0; ax < 3; ++ax) {
                if (q->normal[ax] != (ax == a ? (low ? 1 : -1) : 0)) return FacePlan{};
                if (q->size[ax] != (ax == a ? 1 : d[ax])) return FacePlan{};
                if (q->send_origin[ax] != (ax != a ? 0 : low ? 1 : d[a] - 2)) return FacePlan{};
                if (q->recv_origin[ax] != (ax != a ? 0 : low ? 0 : d[a] - 1)) return FacePlan{};
            }
            if (d[a] < 4) return FacePlan{};
        }
        P.layers[(size_t)c.member] |= 1u << (2 * a + side);
        HOp h[2];
        comm_copies(c, *p, masks(c, 0), masks(c, 1), h);
        for (int k = 0; k < 2; ++k) phase[k][a].push_back(h[k]);
    }
    for (int k = 0; k < 2; ++k)
        if (!merge_phases(phase[k], P.hops[k])) return FacePlan{};
    // The columns of x faces lie a row apart, each in a cache line of its own, so
    // going through them again costs far more than their cells (with copies and
    // layer_alpha_kernel for them too, those took 194 us of the above pair, not
    // 34): pair_kernel exchanges them itself, in the rows that both sides of
    // every x face step this way.
    bool seams = true;
    for (const GroupComm &c : comms) {
        if (!c.normal[0]) continue;
        const size_t m = (size_t)c.member, n = (size_t)c.dst;
        seams = seams && dims[m] == dims[n] && (P.layers[m] >> 2) == (P.layers[n] >> 2);
    }
    size_t bytes = 0;
    std::vector<size_t> at(2 * dims.size(), 0);
    std::vector<int> nb(2 * dims.size(), 0);
    for (const GroupComm &c : comms)
        if (c.normal[0]) nb[2 * (size_t)c.member + (c.normal[0] == 1 ? 0 : 1)] = c.dst;
    for (size_t i = 0; i < dims.size(); ++i)
        for (int side = 0; side < 2; ++side) {
            if (!(P.layers[i] >> side & 1u)) continue;
            const SeamRows R(P.layers[i], dims[i][1], dims[i][2]);
            if (R.ny <= 0 || R.nz <= 0) seams = false;
            at[2 * i + (size_t)side] = bytes;
            bytes += (size_t)kSeamPops * (size_t)std::max(R.count(), 0) * elem;
        }
    if (!seams || bytes == 0 || bytes >= (size_t)1 << 31) return P;
    P.seams = true;
    P.seam_bytes = bytes;
    P.seam_at.swap(at);
    P.seam_nb.swap(nb);
    // the copies in those rows are that kernel's
    for (int k = 0; k < 2; ++k) {
        std::vector<HOp> kept;
        for (const HOp &h : P.hops[k]) {
            const std::array<int, 3> &d = dims[(size_t)h.dm];
            const SeamRows R(P.layers[(size_t)h.dm], d[1], d[2]);
            const int o[3] = {0, R.y0, R.z0}, sz[3] = {d[0], R.ny, R.nz};
            int io[3], is[3];
            if (!box_isect(h.dof, h.sz, o, sz, io, is)) {
                kept.push_back(h);
                continue;
            }
            std::vector<std::array<int, 6>> rest;
            box_minus(h.dof, h.sz, io, is, rest);
            for (const auto &b : rest) kept.push_back(op_at_dst(h, &b[0], &b[3]));
        }
        P.hops[k].swap(kept);
    }
    return P;
}

}  // namespace lbm
