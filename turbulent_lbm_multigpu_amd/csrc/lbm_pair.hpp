// lbm_pair.hpp -- one beta and the alpha that follows it in a single pass over
// the distributions, from one buffer into another.
//
// Two half-steps move each population twice through HBM when every half-step
// is a launch of its own.  Here a work-group walks the planes of an x-y tile:
// beta's results of a plane (halo columns included) go to LDS, alpha takes its
// 19 values from there and stores them once.  Alpha at plane z needs beta's
// results of planes z-1, z and z+1; what it takes from the first two waits in
// registers, so LDS holds two planes (the one being read and the one being
// written) and a plane costs one barrier.  Neighbouring tiles both compute the
// beta of the columns between them: the source buffer is not written, so they
// get the same values.
#pragma once

#include <limits>

#include "lbm_device.hpp"
#include "once_per_device.hpp"
#include "pair_plan.hpp"

namespace lbm {

// The physical parameters of a domain in the compute type, read once: a
// work-group's walk keeps them in scalar registers, with the factors of the
// reference's forcing.
template <typename T>
struct PairPhys {
    T inv_tau, tau0, les_coeff, gx, gy, gz, lid;
    T ref[9];
    int forcing;
};
// A value of uniform bits in scalar registers.  Made opaque first: of a value
// it knows to be uniform the compiler drops the lane read, and leaves it in
// the vector register that a conversion wrote.
__device__ __forceinline__ unsigned scalar_word(unsigned v) {
    asm volatile("" : "+v"(v));
    return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ float scalar_reg(float v) { return __uint_as_float(scalar_word(__float_as_uint(v))); }
__device__ __forceinline__ double scalar_reg(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned long long lo = scalar_word((unsigned)b), hi = scalar_word((unsigned)(b >> 32));
    return __longlong_as_double((long long)((hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ PairPhys<T> pair_phys(const DomDev *D) {
    PairPhys<T> q{scalar_reg((T)D->inv_tau), scalar_reg((T)D->tau0), scalar_reg((T)D->les_coeff),
                  scalar_reg((T)D->gx),      scalar_reg((T)D->gy),   scalar_reg((T)D->gz),
                  scalar_reg((T)D->lid),     {},                     D->forcing};
#pragma unroll
    for (int k = 0; k < 9; ++k) q.ref[k] = scalar_reg(ref_factor<T>(k, (T)D->gx, (T)D->gy, (T)D->gz));
    return q;
}
template <typename T>
__device__ __forceinline__ T ref_forcing(const PairPhys<T> *D, T *f, T rho) {
    return alpha_ref_chain(f, rho, [&](int k) { return D->ref[k]; });
}

// A copy whose values the compiler takes as new: what it derives from them
// (the lid's equilibrium, say) would otherwise be kept in vector registers
// over the whole walk.
template <typename T>
__device__ __forceinline__ PairPhys<T> pair_phys_here(PairPhys<T> q) {
    asm volatile("" : "+s"(q.inv_tau), "+s"(q.tau0), "+s"(q.les_coeff), "+s"(q.lid));
    asm volatile("" : "+s"(q.gx), "+s"(q.gy), "+s"(q.gz));
    return q;
}

// Element access through a buffer descriptor: a lane's byte offset in a
// vector register plus a population's offset in a scalar one, so an address
// costs no vector instruction.  (As global accesses the 38 population bases
// of a walk do not fit the scalar registers, and each access pays a 64-bit
// vector addition.)  A domain's distributions are below 4 GiB.
typedef __amdgpu_buffer_rsrc_t PairBuf;
__device__ __forceinline__ PairBuf pair_buf(gchar *base, unsigned bytes = 0xffffffffu) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)bytes, 0x00020000);
}
template <typename U>
__device__ __forceinline__ U buf_ld(PairBuf b, unsigned off, unsigned pop) {
    if constexpr (sizeof(U) == 4) {
        return (U)__builtin_amdgcn_raw_buffer_load_b32(b, (int)off, (int)pop, 0);
    } else {
        return __builtin_bit_cast(U, __builtin_amdgcn_raw_buffer_load_b64(b, (int)off, (int)pop, 0));
    }
}
template <typename U>
__device__ __forceinline__ void buf_st(PairBuf b, unsigned off, unsigned pop, U v) {
    if constexpr (sizeof(U) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32((unsigned)v, b, (int)off, (int)pop, 0);
    } else {
        typedef unsigned V2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v), b, (int)off, (int)pop, 0);
    }
}

// Column walk of one work-item: byte offsets of the rows y-1, y, y+1 (index 0,
// 1, 2) in the planes z-1, z, z+1 around the plane being gathered.
struct PairRows {
    unsigned o[3][3];  // [plane][row]
    // wavefront-uniform: a lane's x neighbour lies in another layout block
    // (or across the domain's ends), per plane for the rows alpha and beta
    // shift in x: the middle row of every plane, all rows of the middle plane
    bool edge_mid[3], edge_side[3];
};

template <class SP>
__device__ __forceinline__ void pair_plane(PairRows &r, int k, int g, int X, int cells, bool wrap) {
    int idx[3] = {g - X, g, g + X};
    if (wrap) {  // uniform: only the tiles at the domain's ends
#pragma unroll
        for (int q = 0; q < 3; ++q) idx[q] = wrap_idx(idx[q], cells);
        asm volatile("");
    }
    bool e[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        // (idx + 1) & (kBlk - 1) is 0 or 1 at a block's last and first cell
        e[q] = (((unsigned)idx[q] + 1u) & (kBlk - 1u)) < 2u;
        r.o[k][q] = cell_base((unsigned)idx[q]) * SP::kBytes;
    }
    // a wavefront at the domain's ends takes the x neighbours one by one
    r.edge_mid[k] = wrap || __ballot(e[1]) != 0ull;
    r.edge_side[k] = wrap || (__ballot(e[0]) | __ballot(e[2])) != 0ull;
}

// beta's gather of the cell at linear index g (slot opp(i) of g - d_i).  The
// offsets are settled first and every load is issued once, after the branch:
// loads of both branches would meet in copies, and a copy waits for its load.
template <class SP>
__device__ __forceinline__ void pair_gather_cell(PairBuf src, const PairRows &r, int g, int X, int XY, int cells,
                                                 bool wrap, typename SP::U *u) {
    using U = typename SP::U;
    constexpr unsigned es = SP::kBytes;
    unsigned off[19];
#pragma unroll
    for (int i = 0; i < 19; ++i) off[i] = r.o[1 - ez(i)][1 - ey(i)] - (unsigned)ex(i) * es;
    if (r.edge_mid[0] | r.edge_mid[1] | r.edge_mid[2] | r.edge_side[1]) {
#pragma unroll
        for (int i = 0; i < 19; ++i) {
            if (ex(i) == 0) continue;
            int idx = g - (ex(i) + X * ey(i) + XY * ez(i));
            if (wrap) {
                idx = wrap_idx(idx, cells);
                asm volatile("");
            }
            off[i] = cell_base((unsigned)idx) * es;
            asm volatile("" : "+v"(off[i]));  // one at a time: all at once they set the kernel's register count
        }
    }
#pragma unroll
    for (int i = 0; i < 19; ++i) u[i] = buf_ld<U>(src, off[i], (unsigned)opp(i) * kBlk * es);
}

// cell_update of one wavefront, each flag's branch after the other and in
// place: as one chain of alternatives the compiler copies all 19 populations
// at every join.  Fluid wavefronts, nearly all of them, run the first branch
// alone.  Returns whether the cell exchanges its opposite populations on the
// way out against the rest: a beta cell that bounces back, an alpha cell that
// keeps its slots (where the others store f[opp(k)] in slot k); the stores do
// that by their addresses.
template <typename T, bool BETA>
__device__ __forceinline__ bool pair_update(T *f, int flag, const PairPhys<T> &ph, bool macros, T &vx, T &vy, T &vz,
                                            T &dens) {
    if (flag == kFlagFluid) (void)cell_update<T, BETA>(f, kFlagFluid, &ph, vx, vy, vz, dens);
    if (__ballot(flag != kFlagFluid) == 0ull) return false;
    int fl = flag;
    asm volatile("" : "+v"(fl));
    if (fl == kFlagInjection) (void)cell_update<T, BETA>(f, kFlagInjection, &ph, vx, vy, vz, dens);
    int fo = flag;
    asm volatile("" : "+v"(fo));
    if (BETA) return fo == kFlagObstacle;
    const bool keep = fo != kFlagFluid && fo != kFlagInjection;
    // a cell that stores nothing leaves f as it is
    if (macros && keep) (void)cell_update<T, BETA>(f, fo, &ph, vx, vy, vz, dens);
    return keep;
}

// Waits for every vector memory operation issued so far (vmcnt 0; LDS and
// scalar counters untouched).
__device__ __forceinline__ void loads_arrived() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// What bounds it: FP32 with LES issues 1270 vector instructions per cell and
// pair (beta on the halo included; 1070 with 128-cell rows), 91 % (76 %) of the
// SIMDs' issue slots at 256^3; FP64 45 %, with two wavefronts to a SIMD that
// wait for each other's planes.  HBM carries 2.85 GB a pair at 256^3 FP32 where
// two half-step launches move 5.15 GB.  256^3 LES: FP32 336 us a step against 464 in place (419 with the
// best launch shape), FP64 563 against 922 (863).
template <int ST, int NT, bool LAYERS>
__global__ void __launch_bounds__(NT, ST == 1 ? 2 : 4)
    pair_kernel(const DomDev *__restrict__ doms, const PairTile *__restrict__ tiles, void *second, int flip,
                int xcd_map, long long *ctr) {
    using SP = Storage<ST>;
    using T = typename SP::T;
    using U = typename SP::U;
    extern __shared__ char smem[];
    U *const lds = (U *)smem;                                       // beta's values: [2][19][NT]
    uint8_t *const lds_flags = (uint8_t *)smem + 2 * 19 * NT * sizeof(U);  // and flags: [2][NT]
    // the group's half-step counter (see step_kernel): a pair reads one slot and publishes h + 2 in the other
    long long h = 0;
    if (ctr) {
        h = ctr[flip];
        if (blockIdx.x == 0 && threadIdx.x == 0) ctr[flip ^ 1] = h + 2;
    }
    const int nb = (int)gridDim.x;
    const int t = xcd_map < 0   ? xcd_tile((int)blockIdx.x, nb)
                  : xcd_map > 0 ? xcd_chunk_tile((int)blockIdx.x, nb, xcd_map)
                                : (int)blockIdx.x;
    const PairTile P = tiles[t];
    const DomDev *D = doms + P.dom;
    if (h >= D->stop_at) return;  // uniform: before any barrier
    const PairPhys<T> phys = pair_phys<T>(D);
    const bool macros = D->store_velocity || D->store_density;
    const int X = D->nx, XY = D->nx * D->ny, cells = (int)D->cells;
    // Lanes past the tile's columns run along on a column of it (beta on its
    // first, with an LDS position of their own; alpha on its first inner one,
    // storing nothing), so the walk has no lane-dependent branch around its
    // loads.  A wavefront without columns only keeps the barriers.
    PairLane LB = pair_beta_lane(P, X, (int)threadIdx.x), LA = pair_alpha_lane(P, X, (int)threadIdx.x);
    const int z0 = P.z0, nz = P.nz;
    if (__ballot(LB.pos >= 0) == 0ull) {
        for (int k = 0; k < nz + 2; ++k) __syncthreads();
        return;
    }
    if (LB.pos < 0) LB = PairLane{(int)threadIdx.x, P.org};
    const bool stores = LA.pos >= 0;
    const int alpha_from = (int)scalar_word(__ballot(stores) != 0ull ? 2u : (unsigned)nz + 2u);  // first plane of the walk with an alpha
    if (!stores) LA = pair_alpha_lane(P, X, 0);
    const int pitch = pair_pitch(P, X);
    // Cells whose alpha has to wait for an exchange keep beta's values.  Over an
    // x face, the inner cell's alpha takes what comes in from `seam` and goes to
    // the ghost cell beyond the face, whose own lane leaves those slots out.
    bool waits = false, inner[2] = {false, false}, ghost[2] = {false, false};
    unsigned seam_at = 1u << 31;  // past the buffer: nothing is fetched
    gchar *beyond = nullptr;
    const SeamRows SR(D->layers, D->ny, D->nz);
    if constexpr (LAYERS) {
        const int y = LA.p / X, x = LA.p - y * X, side = x >= 2;
        const bool face = in_layers(D->layers, 0, x, X), rim = in_layers(D->layers, 1, y, D->ny);
        waits = rim || (face && !D->seam);
        if (face && !waits) {
            const bool out = x == (side ? X - 1 : 0);
            inner[side] = !out;
            ghost[side] = out;
            if (!out) {
                const DomDev *N = doms + D->seam_nb[side];
                beyond = (gchar *)(flip ? N->dd : N->dd2);
                seam_at = D->seam_at[side] + (unsigned)(y - SR.y0) * SP::kBytes;
            }
        }
    }
    void *const two = second ? second : D->dd2;
    gchar *const from = (gchar *)(flip ? two : D->dd);
    const PairBuf dst = pair_buf((gchar *)(flip ? D->dd : two));
    const guchar *const flags = (const guchar *)D->flags;
    const bool wrap = pair_wraps(P, X, XY, cells);
    int g = LB.p + XY * (z0 - 1);  // the cell whose populations are loaded next
    PairRows rows{};
    U u[19];
    int flag_next;
    auto load = [&](unsigned bytes) {
        pair_gather_cell<SP>(pair_buf(from, bytes), rows, g, X, XY, cells, wrap, u);
        int idx = g;
        if (wrap) {
            idx = wrap_idx(idx, cells);
            asm volatile("");
        }
        flag_next = (int)flags[(unsigned)idx];
    };
    // beta of the plane in u, into LDS; then the next plane's loads, which are
    // in flight during the barrier and alpha.  After the last plane they are
    // out of the descriptor's range and fetch nothing (skipped by a branch,
    // they would meet in copies that wait for them).
    auto beta_plane = [&](int k) {
        U *const buf = lds + (k & 1) * 19 * NT + LB.pos;
        T f[19], vx, vy, vz, dens;
        const int flag = flag_next;
#pragma unroll
        for (int i = 0; i < 19; ++i) f[i] = kin<SP>(u[i], i);
        const PairPhys<T> ph = pair_phys_here(phys);
        const bool bounce = pair_update<T, true>(f, flag, ph, false, vx, vy, vz, dens);
        U *const even = buf + (bounce ? NT : 0), *const odd = buf + (bounce ? 0 : NT);
#pragma unroll
        for (int i = 0; i < 18; i += 2) {
            even[i * NT] = kout<SP>(f[i], i);
            odd[i * NT] = kout<SP>(f[i + 1], i + 1);
        }
        buf[18 * NT] = kout<SP>(f[18], 18);
        lds_flags[(k & 1) * NT + LB.pos] = (uint8_t)flag;
        asm volatile("" ::: "memory");  // the loads below take f's registers
        g += XY;
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
            rows.o[0][dy] = rows.o[1][dy];
            rows.o[1][dy] = rows.o[2][dy];
        }
        rows.edge_mid[0] = rows.edge_mid[1];
        rows.edge_mid[1] = rows.edge_mid[2];
        rows.edge_side[1] = rows.edge_side[2];
        pair_plane<SP>(rows, 2, g + XY, X, cells, wrap);
        load(scalar_word(k < nz + 1 ? 0xffffffffu : 0u));
        __syncthreads();
    };
    // beta values waiting for alpha: of the plane before (ez = 0 and the rest
    // population, with the flag) and of the two planes before (ez = +1)
    U mid[9], up0[5], up1[5];
    int flag_mid;
    auto at = [&](int k, int i) {
        return lds[((k & 1) * 19 + i) * NT + LA.pos - (ex(i) + pitch * ey(i))];
    };
    auto take_plane = [&](int k) {
        int q0 = 0, qu = 0;
#pragma unroll
        for (int i = 0; i < 19; ++i) {
            if (ez(i) == 0) mid[q0++] = at(k, i);
            if (ez(i) > 0) {
                up1[qu] = up0[qu];
                up0[qu] = at(k, i);
                ++qu;
            }
        }
        flag_mid = lds_flags[(k & 1) * NT + LA.pos];
    };
#pragma unroll
    for (int q = 0; q < 5; ++q) up0[q] = 0;
    pair_plane<SP>(rows, 0, g - XY, X, cells, wrap);
    pair_plane<SP>(rows, 1, g, X, cells, wrap);
    pair_plane<SP>(rows, 2, g + XY, X, cells, wrap);
    load(0xffffffffu);
    loads_arrived();
    int k = 0;
    for (; k < alpha_from; ++k) {
        beta_plane(k);
        loads_arrived();
        take_plane(k);
    }
    for (; k < nz + 2; ++k) {
        const int z = z0 + k - 2;
        const bool rows_z = z >= SR.z0 && z < SR.z0 + SR.nz;
        U in[kSeamPops];
        if constexpr (LAYERS) {
            const PairBuf sb = pair_buf((gchar *)D->seam, scalar_word(rows_z && D->seam ? D->seam_bytes : 0u));
            const unsigned at_row = seam_at + (unsigned)((z - SR.z0) * SR.ny) * SP::kBytes;
#pragma unroll
            for (int q = 0; q < kSeamPops; ++q) in[q] = buf_ld<U>(sb, at_row, (unsigned)(q * SR.count()) * SP::kBytes);
        }
        beta_plane(k);
        T f[19], vx, vy, vz, dens;
        int q0 = 0, qu = 0;
#pragma unroll
        for (int i = 0; i < 19; ++i) {
            const U v = ez(i) == 0 ? mid[q0] : ez(i) > 0 ? up1[qu] : at(k, i);
            if (ez(i) == 0) ++q0;
            if (ez(i) > 0) ++qu;
            f[i] = kin<SP>(v, i);
        }
        const PairPhys<T> ph = pair_phys_here(phys);
        int flag = flag_mid;
        if constexpr (LAYERS) {
            if (waits || !rows_z) flag = kFlagGhost;  // a ghost cell's values pass
            int q = 0;
#pragma unroll
            for (int i = 0; i < 18; i += 2) {  // ex(i) = 1 comes with ex(i + 1) = -1
                if (ex(i) == 0) continue;
                const T v = kin<SP>(in[q], i);
                f[i] = inner[0] && rows_z ? v : f[i];
                f[i + 1] = inner[1] && rows_z ? v : f[i + 1];
                ++q;
            }
        }
        const bool keep = pair_update<T, false>(f, flag, ph, macros, vx, vy, vz, dens);
        // The next plane's loads are waited for before the stores: at the top
        // of the next plane the wait would cover the stores as well.
        loads_arrived();
        if (stores) {
            const unsigned gs = (unsigned)(LA.p + XY * z);
            const unsigned own = cell_base(gs) * SP::kBytes;
            constexpr unsigned pop = kBlk * SP::kBytes;
            const unsigned even = own + (keep ? 0u : pop), odd = own + (keep ? pop : 0u);
            auto put = [&](bool along_x, bool evens, bool odds) {
#pragma unroll
                for (int i = 0; i < 18; i += 2) {
                    if ((ex(i) != 0) != along_x) continue;
                    if (evens) buf_st<U>(dst, even, (unsigned)i * pop, kout<SP>(f[i], i));
                    if (odds) buf_st<U>(dst, odd, (unsigned)i * pop, kout<SP>(f[i + 1], i + 1));
                }
            };
            if constexpr (LAYERS) {
                const bool low = ghost[0] && rows_z, high = ghost[1] && rows_z;
                if (!((low || high) && D->seam_all)) {
                    put(false, true, true);
                    buf_st<U>(dst, own, 18u * pop, kout<SP>(f[18], 18));
                    // the low ghost cell leaves the slots with ex = -1 out, the high one those with ex = 1
                    if (!(keep ? high : low)) put(true, true, false);
                    if (!(keep ? low : high)) put(true, false, true);
                }
                if ((inner[0] || inner[1]) && rows_z) {
                    const int to = inner[0] ? X - 2 : 2 - X;
                    gchar *const n = beyond + (size_t)(cell_base(gs + (unsigned)to) * SP::kBytes);
                    const bool all = D->seam_all;
#pragma unroll
                    for (int i = 0; i < 18; i += 2) {
                        const U a = kout<SP>(keep ? f[i] : f[i + 1], i), b = kout<SP>(keep ? f[i + 1] : f[i], i + 1);
                        if (all || (ex(i) != 0 && inner[0])) raw_st<false, U>(n + (size_t)i * pop, 0u, a);
                        if (all || (ex(i) != 0 && inner[1])) raw_st<false, U>(n + (size_t)(i + 1) * pop, 0u, b);
                    }
                    if (all) raw_st<false, U>(n + (size_t)18 * pop, 0u, kout<SP>(f[18], 18));
                }
            } else {
#pragma unroll
                for (int i = 0; i < 18; i += 2) {
                    buf_st<U>(dst, even, (unsigned)i * pop, kout<SP>(f[i], i));
                    buf_st<U>(dst, odd, (unsigned)i * pop, kout<SP>(f[i + 1], i + 1));
                }
                buf_st<U>(dst, own, 18u * pop, kout<SP>(f[18], 18));
            }
            if (macros && flag != kFlagGhost) store_macros<T>(D, gs, cells, vx, vy, vz, dens);
        }
        take_plane(k);
    }
}

// Alpha of the layers that pair_kernel left at beta's values, after their
// exchange: `boxes` and, per block, the box it belongs to.  Bound by memory, as
// alpha of a whole domain: 262,144 cells of y and z layers, FP32, in 13 us.
template <int ST>
__global__ void __launch_bounds__(256)
    layer_alpha_kernel(const DomDev *__restrict__ doms, const LayerBox *__restrict__ boxes,
                       const int *__restrict__ block_box, int flip) {
    using SP = Storage<ST>;
    using T = typename SP::T;
    using U = typename SP::U;
    const LayerBox &B = boxes[block_box[blockIdx.x]];
    const DomDev *D = doms + B.dom;
    const int e = ((int)blockIdx.x - B.block_begin) * 256 + (int)threadIdx.x;
    if (e >= B.s[0] * B.s[1] * B.s[2]) return;
    const int r = e / B.s[0], bz = r / B.s[1];
    const int x = B.o[0] + e - r * B.s[0], y = B.o[1] + r - bz * B.s[1], z = B.o[2] + bz;
    if (B.axis < 2 && in_layers(D->layers, 2, z, D->nz)) return;
    if (B.axis < 1 && in_layers(D->layers, 1, y, D->ny)) return;
    const unsigned g = (unsigned)(x + D->nx * (y + D->ny * z));
    const int flag = (int)((const guchar *)D->flags)[g];
    if (flag == kFlagGhost) return;
    gchar *const own = (gchar *)(flip ? D->dd : D->dd2) + (size_t)cell_base(g) * SP::kBytes;
    constexpr size_t pop = (size_t)kBlk * SP::kBytes;
    T f[19], vx, vy, vz, dens;
#pragma unroll
    for (int i = 0; i < 19; ++i) f[i] = kin<SP>(raw_ld<false, U>(own + i * pop, 0u), i);
    if (cell_update<T, false>(f, flag, D, vx, vy, vz, dens)) {
#pragma unroll
        for (int k = 0; k < 19; ++k) raw_st<false, U>(own + k * pop, 0u, kout<SP>(f[opp(k)], k));
    }
    store_macros<T>(D, g, (int)D->cells, vx, vy, vz, dens);
}

// What beta of the domain beyond an x face moves over it, into the seam buffer
// for the pair of this domain: beta of the column next to its ghost layer, from
// the buffer the pair starts in.  Bound by cache lines, 19 for a cell: 131,072
// cells, FP32, in 89 us (3.6 TB/s of lines).  The alternative, pair_kernel
// leaving both layers of a face by rows and a kernel after it doing their alpha
// and exchange, stores single columns twice: 52 us more in pair_kernel, 82 in
// that kernel.
template <int ST>
__global__ void __launch_bounds__(256)
    seam_beta_kernel(const DomDev *__restrict__ doms, const SeamFace *__restrict__ faces,
                     const int *__restrict__ block_face, int flip) {
    using SP = Storage<ST>;
    using T = typename SP::T;
    using U = typename SP::U;
    const SeamFace F = faces[block_face[blockIdx.x]];
    const DomDev *N = doms + F.nb;
    const int X = N->nx, XY = X * N->ny, cells = (int)N->cells;
    const SeamRows SR(N->layers, N->ny, N->nz);  // those of both sides
    // the rows whose populations reach such a row; past the ends by the linear wrap
    const int wy = SR.ny + 2, e = ((int)blockIdx.x - F.block_begin) * 256 + (int)threadIdx.x;
    if (e >= wy * (SR.nz + 2)) return;
    const int rz = e / wy, y = SR.y0 - 1 + e - rz * wy, z = SR.z0 - 1 + rz;
    const int g = (F.side ? 1 : X - 2) + X * y + XY * z;
    PairRows rows;
    pair_plane<SP>(rows, 0, g - XY, X, cells, true);
    pair_plane<SP>(rows, 1, g, X, cells, true);
    pair_plane<SP>(rows, 2, g + XY, X, cells, true);
    U u[19];
    pair_gather_cell<SP>(pair_buf((gchar *)(flip ? N->dd2 : N->dd)), rows, g, X, XY, cells, true, u);
    const int flag = (int)((const guchar *)N->flags)[(unsigned)wrap_idx(g, cells)];
    T f[19], vx, vy, vz, dens;
#pragma unroll
    for (int i = 0; i < 19; ++i) f[i] = kin<SP>(u[i], i);
    const PairPhys<T> ph = pair_phys_here(pair_phys<T>(N));
    const bool bounce = pair_update<T, true>(f, flag, ph, false, vx, vy, vz, dens);
    gchar *const to = (gchar *)N->seam + doms[F.dom].seam_at[F.side];
    int q = 0;
#pragma unroll
    for (int i = 0; i < 18; i += 2) {
        if (ex(i) == 0) continue;
        // the one of the two that moves to this domain: ex = 1 over its low face
        const bool first = F.side == 0;
        const int ty = y + (first ? ey(i) : ey(i + 1)), tz = z + (first ? ez(i) : ez(i + 1));
        const T v = first != bounce ? f[i] : f[i + 1];
        if (SR.has(ty, tz))
            raw_st<false, U>(to + ((size_t)q * SR.count() + (ty - SR.y0) + (size_t)(tz - SR.z0) * SR.ny) * SP::kBytes,
                             0u, kout<SP>(v, i));
        ++q;
    }
}

// The two sizes of the small-domain kernel: cells (halo included) its LDS
// holds, and its work-items.  The small one takes a box in one pass; the large
// one fills the 160 KB of LDS.
constexpr int kBoxSmall = 704;
constexpr int box_large(int storage) { return storage == 1 ? 1056 : 2048; }
constexpr int box_threads(int storage) { return storage == 1 ? 512 : 1024; }

// The pair of a small domain: a work-group computes the beta of a whole box,
// halo included, into LDS, and after one barrier the alpha of its inner cells.
// Small domains are bound by what a launch costs (about 4 us of dispatch,
// first loads and drain, whatever the kernel does); this halves their number,
// at the price of the beta on the halo (1.8 to 3 times the inner cells).
template <int ST, int NT, int CELLS>
__global__ void __launch_bounds__(NT)
    pair_box_kernel(const DomDev *__restrict__ doms, const PairTile *__restrict__ tiles, void *second, int flip,
                    int xcd_map, long long *ctr) {
    using SP = Storage<ST>;
    using T = typename SP::T;
    using U = typename SP::U;
    extern __shared__ char smem[];
    U *const lds = (U *)smem;                                     // beta's values: [19][CELLS]
    uint8_t *const lds_flags = (uint8_t *)smem + 19 * CELLS * sizeof(U);  // and flags: [CELLS]
    long long h = 0;  // as in pair_kernel
    if (ctr) {
        h = ctr[flip];
        if (blockIdx.x == 0 && threadIdx.x == 0) ctr[flip ^ 1] = h + 2;
    }
    const int nb = (int)gridDim.x;
    const int t = xcd_map < 0 ? xcd_tile((int)blockIdx.x, nb) : (int)blockIdx.x;
    const PairTile P = tiles[t];
    const DomDev *D = doms + P.dom;
    if (h >= D->stop_at) return;  // uniform: before any barrier
    const PairPhys<T> phys = pair_phys<T>(D);
    const bool macros = D->store_velocity || D->store_density;
    const int X = D->nx, XY = D->nx * D->ny, cells = (int)D->cells;
    void *const two = second ? second : D->dd2;
    const PairBuf src = pair_buf((gchar *)(flip ? two : D->dd)), dst = pair_buf((gchar *)(flip ? D->dd : two));
    const guchar *const flags = (const guchar *)D->flags;
    const bool wrap = pair_wraps(P, X, XY, cells);
    const int w = P.w, wh = P.w * P.h, n = wh * (P.nz + 2);
    for (int e = (int)threadIdx.x; e < n; e += NT) {
        const int tz = e / wh, r = e - tz * wh, ty = r / w;
        const int g = P.org + r - ty * w + X * ty + XY * (P.z0 - 1 + tz);
        PairRows rows;
        pair_plane<SP>(rows, 0, g - XY, X, cells, wrap);
        pair_plane<SP>(rows, 1, g, X, cells, wrap);
        pair_plane<SP>(rows, 2, g + XY, X, cells, wrap);
        U u[19];
        pair_gather_cell<SP>(src, rows, g, X, XY, cells, wrap, u);
        const int flag = (int)flags[(unsigned)(wrap ? wrap_idx(g, cells) : g)];
        T f[19], vx, vy, vz, dens;
#pragma unroll
        for (int i = 0; i < 19; ++i) f[i] = kin<SP>(u[i], i);
        const PairPhys<T> ph = pair_phys_here(phys);
        const bool bounce = pair_update<T, true>(f, flag, ph, false, vx, vy, vz, dens);
        U *const even = lds + e + (bounce ? CELLS : 0), *const odd = lds + e + (bounce ? 0 : CELLS);
#pragma unroll
        for (int i = 0; i < 18; i += 2) {
            even[i * CELLS] = kout<SP>(f[i], i);
            odd[i * CELLS] = kout<SP>(f[i + 1], i + 1);
        }
        lds[18 * CELLS + e] = kout<SP>(f[18], 18);
        lds_flags[e] = (uint8_t)flag;
    }
    __syncthreads();
    const int iw = P.w - 2, iwh = iw * (P.h - 2), ni = iwh * P.nz;
    for (int e = (int)threadIdx.x; e < ni; e += NT) {
        const int tz = e / iwh, r = e - tz * iwh, ty = r / iw, tx = r - ty * iw;
        const int pos = (tz + 1) * wh + (ty + 1) * w + tx + 1;
        T f[19], vx, vy, vz, dens;
#pragma unroll
        for (int i = 0; i < 19; ++i) f[i] = kin<SP>(lds[i * CELLS + pos - (ex(i) + w * ey(i) + wh * ez(i))], i);
        const int flag = lds_flags[pos];
        const PairPhys<T> ph = pair_phys_here(phys);
        const bool keep = pair_update<T, false>(f, flag, ph, macros, vx, vy, vz, dens);
        const unsigned gs = (unsigned)(P.org + tx + 1 + X * (ty + 1) + XY * (P.z0 + tz));
        const unsigned own = cell_base(gs) * SP::kBytes;
        constexpr unsigned pop = kBlk * SP::kBytes;
        const unsigned even = own + (keep ? 0u : pop), odd = own + (keep ? pop : 0u);
#pragma unroll
        for (int i = 0; i < 18; i += 2) {
            buf_st<U>(dst, even, (unsigned)i * pop, kout<SP>(f[i], i));
            buf_st<U>(dst, odd, (unsigned)i * pop, kout<SP>(f[i + 1], i + 1));
        }
        buf_st<U>(dst, own, 18u * pop, kout<SP>(f[18], 18));
        if (macros && flag != kFlagGhost) store_macros<T>(D, gs, cells, vx, vy, vz, dens);
    }
}

// Calls f(kernel, work-items, bytes of LDS) with the kernel of a launch.
template <int ST, class F>
hipError_t with_pair_kernel(const PairLaunch &L, F &&f) {
    constexpr int per_cell = 19 * (int)Storage<ST>::kBytes + 1;
    constexpr int NT = ST == 1 ? 512 : 1024;
    constexpr int NB = box_threads(ST), CB = box_large(ST);
    if (L.box_cells == kBoxSmall) return f(pair_box_kernel<ST, kBoxSmall, kBoxSmall>, kBoxSmall, kBoxSmall * per_cell);
    if (L.box_cells == CB) return f(pair_box_kernel<ST, NB, CB>, NB, CB * per_cell);
    if (L.box_cells > 0) return hipErrorInvalidValue;
    if (L.layers) return f(pair_kernel<ST, NT, true>, NT, 2 * NT * per_cell);
    return f(pair_kernel<ST, NT, false>, NT, 2 * NT * per_cell);
}

// Lets the kernel of a launch use its LDS, on the current device: the
// attribute belongs to the function as it is loaded there.
template <int ST>
hipError_t allow_pair_lds(const PairLaunch &L, int device) {
    static OncePerDevice once;
    return with_pair_kernel<ST>(L, [&](auto *kernel, int, int lds) -> hipError_t {
        hipError_t e = hipSuccess;
        once((const void *)kernel, device, [&] {
            e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            return e == hipSuccess;
        });
        return e;
    });
}

// Launch of a pair kernel: beta and alpha of every tile from one buffer into
// the other (flip 0: from dd, 1: back into it).  `second`: the second buffer
// of a single domain, or null for the one its descriptor names.
template <int ST>
hipError_t launch_pair_storage(const PairLaunch &L, int ntiles, const DomDev *descs, const PairTile *tiles,
                               void *second, hipStream_t stream, long long *ctr, int flip) {
    return with_pair_kernel<ST>(L, [&](auto *kernel, int threads, int lds) -> hipError_t {
        if (L.threads != threads) return hipErrorInvalidValue;
        kernel<<<ntiles, threads, lds, stream>>>(descs, tiles, second, flip, L.xcd_map, ctr);
        return hipGetLastError();
    });
}

}  // namespace lbm
