// Per-cell device code of the A-A step shared by the single-domain kernels
// (lbm_step.hip) and the multi-cavity batch kernels (lbm_batch.hip):
// population accessors, one cell of alpha and of beta, fused x-face packing.
#pragma once

#include "lbm_d3q19.hpp"
#include "lbm_internal.hpp"
#include "lbm_storage.hpp"

namespace lbm {


constexpr int kBlock = 256;

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2). Renumber them so every XCD works on one contiguous range of cells:
// neighbouring cells then share partial cache lines inside one L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb)
{
    const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u, k = b >> 3;
    return x * q + (x < r ? x : r) + k;
}

// The block of cells that this workgroup steps.
template <class C>
__device__ __forceinline__ uint32_t step_block(const StepArgs<C>& a)
{
    const uint32_t b = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    return a.reverse ? gridDim.x - 1 - b : b;
}

template <class C>
__device__ __forceinline__ uint32_t box_cell(const StepArgs<C>& a, uint32_t gid)
{
    const uint32_t t = a.div_bx.div(gid);
    const uint32_t x = gid - t * a.div_bx.d;
    const uint32_t z = a.div_by.div(t);
    const uint32_t y = t - z * a.div_by.d;
    return (uint32_t)((a.oz + (int32_t)z) * a.nxy + (a.oy + (int32_t)y) * a.nx + a.ox + (int32_t)x);
}

// Population accessors. Acc32 keeps one uniform base pointer per plane (the
// beta neighbour shift is folded into it) and one 32-bit byte offset per lane
// shared by all 19 planes, so every access is a saddr global load/store with
// no per-plane vector address arithmetic; it needs cells * sizeof(S) < 2^32.
// AccWrap32 serves the same planes where the reference's linear-index wrap
// (domainWrap, CLbmBetaCPU.cpp:44-50) may apply: a uniform unshifted base and
// a wrapped 32-bit offset per plane. Acc64 uses a 64-bit element index per
// plane, with WRAP the wrap as well.
// for_stores() gives the accessor a step's stores go through: a fresh (empty
// asm) copy of the lane's offset or index, from which the addresses are formed
// anew. Without it the compiler keeps the loads' addresses live across the
// collision: 19 VGPR pairs, or 38 VGPRs of wrapped indices.
// The plane bases come precomputed in the kernel arguments: opaque uniform
// values the compiler cannot fold into per-lane pointer chains.
// Every population array is device (global) memory. The accessors say so
// explicitly: a base pointer read from memory (the batch member tables) is
// otherwise a generic pointer, and generic accesses compile to flat
// instructions, which wait on both memory counters.
#define LBM_GLOBAL __attribute__((address_space(1)))

template <class T>
__device__ __forceinline__ T fresh(T v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// outputs() stores a cell's rho and u where the solver keeps them.
struct CellOutputs {
    template <class C>
    __device__ __forceinline__ void outputs(const StepArgs<C>& a, uint32_t id, C rho, C ux, C uy,
                                            C uz) const
    {
        if (a.store_u) {
            a.u[id] = ux;
            a.u[a.stride + id] = uy;
            a.u[2 * a.stride + id] = uz;
        }
        if (a.store_rho)
            a.rho[id] = rho;
    }
};

template <class S, bool NT>
struct Acc32 : CellOutputs {
    __device__ __forceinline__ Acc32(const char* const* p, uint32_t o) : plane(p), off(o) {}
    const char* const* plane;
    uint32_t off;
    __device__ __forceinline__ Acc32 for_stores() const { return {plane, fresh(off)}; }
    __device__ __forceinline__ S load(int l, int32_t) const
    {
        const LBM_GLOBAL S* p = (const LBM_GLOBAL S*)(plane[l] + off);
        if (NT)
            return __builtin_nontemporal_load(p);
        return *p;
    }
    __device__ __forceinline__ void store(int l, int32_t, S v) const
    {
        LBM_GLOBAL S* p = (LBM_GLOBAL S*)(const_cast<char*>(plane[l]) + off);
        if (NT)
            __builtin_nontemporal_store(v, p);
        else
            *p = v;
    }
};

// id + delta wrapped into [0, n) once, as the reference does.
__device__ __forceinline__ int32_t wrapped(int32_t id, int32_t delta, int32_t n)
{
    int32_t j = id + delta;
    j = (j >= n) ? j - n : j;
    return (j < 0) ? j + n : j;
}

template <class S>
struct AccWrap32 : CellOutputs {
    __device__ __forceinline__ AccWrap32(const char* d, int64_t st, int32_t i, int32_t cells)
        : dd(d), stride(st), id(i), n(cells)
    {
    }
    const char* dd;
    int64_t stride;
    int32_t id, n;
    __device__ __forceinline__ AccWrap32 for_stores() const { return {dd, stride, fresh(id), n}; }
    __device__ __forceinline__ S load(int l, int32_t delta) const
    {
        const char* base = dd + (int64_t)l * stride * (int64_t)sizeof(S);
        return *(const LBM_GLOBAL S*)(base + (uint32_t)wrapped(id, delta, n) * (uint32_t)sizeof(S));
    }
    __device__ __forceinline__ void store(int l, int32_t delta, S v) const
    {
        char* base = const_cast<char*>(dd) + (int64_t)l * stride * (int64_t)sizeof(S);
        *(LBM_GLOBAL S*)(base + (uint32_t)wrapped(id, delta, n) * (uint32_t)sizeof(S)) = v;
    }
};

template <class S, bool WRAP>
struct Acc64 : CellOutputs {
    __device__ __forceinline__ Acc64(S* d, int64_t st, int32_t i, int32_t cells)
        : dd(d), stride(st), id(i), n(cells)
    {
    }
    S* dd;
    int64_t stride;
    int32_t id, n;
    __device__ __forceinline__ Acc64 for_stores() const { return {dd, stride, fresh(id), n}; }
    __device__ __forceinline__ int64_t index(int l, int32_t delta) const
    {
        return (int64_t)l * stride + (WRAP ? wrapped(id, delta, n) : id + delta);
    }
    __device__ __forceinline__ S load(int l, int32_t delta) const
    {
        return ((const LBM_GLOBAL S*)dd)[index(l, delta)];
    }
    __device__ __forceinline__ void store(int l, int32_t delta, S v) const
    {
        ((LBM_GLOBAL S*)dd)[index(l, delta)] = v;
    }
};

// ------------------------------------------------------- fused x packing ---

// Whether the cell lies in the LEFT (x = 1) / RIGHT (x = nx - 2) send plane
// with a fused pack (pl / pr) or unpack (ul / ur) buffer on that side;
// row = z * ny + y is its index in the dense face buffers. Returns pl || pr.
template <class C>
__device__ __forceinline__ bool xpack_where(const StepArgs<C>& a, uint32_t id, uint32_t& row,
                                            bool& pl, bool& pr, bool& ul, bool& ur)
{
    pl = pr = ul = ur = false;
    row = 0;
    if (!a.xpack_on)
        return false;
    row = a.div_nx.div(id);
    const int x = (int)(id - row * (uint32_t)a.nx);
    pl = x == 1 && a.xpack[0] != nullptr;
    pr = x == a.nx - 2 && a.xpack[1] != nullptr;
    ul = x == 1 && a.xunpack[0] != nullptr;
    ur = x == a.nx - 2 && a.xunpack[1] != nullptr;
    return pl || pr;
}

// After alpha: the slot values of a send-plane cell that the neighbour's halo
// needs, the planes whose vectors point back into this solver (c_x = +1 on the
// LEFT send plane, c_x = -1 on the RIGHT one), in the layout lbm_pack_face
// writes ([slot][row]); values pass through the storage type so 16-bit storage
// packs exactly what was stored.
template <class P>
__device__ __forceinline__ void xpack_alpha(const StepArgs<typename P::C>& a, uint32_t row,
                                            bool pl, bool pr, const typename P::C (&v)[kQ])
{
#pragma unroll
    for (int s = 0; s < kQ - 1; s++) {
        if (cx(s) == 0 || !(cx(s) > 0 ? pl : pr))
            continue;
        a.xpack[cx(s) > 0 ? 0 : 1][(int64_t)s * a.fcells + row] = P::load(P::store(v[s], s), s);
    }
}

// After beta: the populations that cross the x faces. From a LEFT send-plane
// cell the directions with c_x = -1 land in the LEFT halo plane, from a RIGHT
// one those with c_x = +1 land in the RIGHT halo plane; each is written at
// its landing cell's row (reference linear wrap), i.e. exactly the entries
// of the halo-plane pack that the neighbour's direction-filtered unpack reads.
template <class P>
__device__ __forceinline__ void xpack_beta(const StepArgs<typename P::C>& a, uint32_t row,
                                           bool pl, bool pr, const typename P::C (&v)[kQ])
{
#pragma unroll
    for (int l = 0; l < kQ - 1; l++) {
        const bool side = cx(l) < 0 ? pl : (cx(l) > 0 ? pr : false);
        if (cx(l) != 0 && side) {
            int32_t t = (int32_t)row + cy(l) + cz(l) * a.ny;
            t = t < 0 ? t + a.fcells : t;
            t = t >= a.fcells ? t - a.fcells : t;
            a.xpack[cx(l) < 0 ? 0 : 1][(int64_t)l * a.fcells + t] = P::load(P::store(v[l], l), l);
        }
    }
}

// ------------------------------------------------------ fused x unpacking ---

// The face work compiled into a step kernel: none, the fused x-face pack
// (lbm_set_step_pack), or the pack and the fused x-face unpack
// (lbm_set_step_unpack); a kernel without a part carries none of its code.
constexpr int kXfNone = 0, kXfPack = 1, kXfUnpack = 2;

// A received x-face buffer brings one plane of each opposite pair
// (xplane(k), xplane(k) + 1) = (c_x = +1, c_x = -1), k = 0..4: before alpha
// the send-plane cell's own slots of the vectors pointing into the solver
// through its face (c_x = +1 on the LEFT send plane, -1 on the RIGHT one:
// what lbm_unpack_face(phase 1) stores there); before beta the halo-plane
// slots the cell reads (c_x = -1 in the LEFT halo plane, +1 in the RIGHT one:
// what lbm_unpack_face(phase 0) stores there). `odd` selects the c_x = -1
// plane of each pair. Opposite vectors share their lattice weight, so both
// planes of a pair decode with xplane(k).
__host__ __device__ constexpr int xplane(int k) { return k == 0 ? 0 : 2 * k + 2; }

// The plane of each pair a face cell receives: before alpha (STEP 0) the
// LEFT face brings c_x = +1 and the RIGHT face c_x = -1, before beta the
// reverse.
template <int STEP>
__device__ __forceinline__ int xunpack_odd(bool ul)
{
    return STEP == 0 ? (ul ? 0 : 1) : (ul ? 1 : 0);
}

// Loads a face cell's 5 received values (ul: from the LEFT buffer, else the
// RIGHT one), issued with its slot loads. A beta cell's halo slots sit at the
// rows of their halo-plane cells (the reference linear wrap, as in
// xpack_beta).
template <class P, int STEP>
__device__ __forceinline__ void xunpack_load(const StepArgs<typename P::C>& a, uint32_t row,
                                             bool ul, int odd, typename P::C (&u)[5])
{
    const typename P::C* buf = a.xunpack[ul ? 0 : 1];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const int e = xplane(k);
        int32_t t = (int32_t)row;
        if (STEP == 1) {
            const int32_t off = cy(e) + cz(e) * a.ny;   // the c_x = -1 plane's is -off
            t += odd ? -off : off;
            t = t < 0 ? t + a.fcells : t;
            t = t >= a.fcells ? t - a.fcells : t;
        }
        u[k] = buf[(int64_t)(e + odd) * a.fcells + t];
    }
}

// The value a step would load from the slot after lbm_unpack_face: the
// received one through the storage type, its range marked in ov as the
// unpack marks it.
template <class P>
__device__ __forceinline__ typename P::C xunpack_value(typename P::C r, int l, uint32_t& ov)
{
    return P::load(P::store_checked(r, l, ov), l);
}

// -------------------------------------------------------------- collision ---

// Both directions of an opposite pair with velocity +-v and weight w, the
// equilibria of common.h:132-160: w * (rho + (+-3 v) + 4.5 v^2). -3 v is
// exactly -(3 v), so the pair shares 3 v and 4.5 v^2 with every result's bits
// kept; with the 16-bit formats and with domains that stay in the Infinity
// Cache the steps are as much bound by instructions as by memory.
template <class C>
__device__ __forceinline__ void equilibrium_pair(C& fp, C& fm, C rho, C v, C w)
{
    const C t = (C)3 * v, q = ((C)9 / (C)2) * (v * v);
    fp = w * ((rho + t) + q);
    fm = w * ((rho - t) + q);
}

// Applies op(direction, opposite, velocity, weight) to the nine opposite pairs,
// one after the other: few values live beside the 19 populations.
template <class C, class Op>
__device__ __forceinline__ void for_pairs(C ux, C uy, C uz, Op op)
{
    constexpr C wa = (C)1 / (C)18, wd = (C)1 / (C)36;
    op(0, 1, ux, wa);
    op(2, 3, uy, wa);
    op(4, 5, ux + uy, wd);
    op(6, 7, ux - uy, wd);
    op(8, 9, ux + uz, wd);
    op(10, 11, ux - uz, wd);
    op(12, 13, uy + uz, wd);
    op(14, 15, uy - uz, wd);
    op(16, 17, uz, wa);
}

// d += inv_tau * (eq - d) in every direction; terms(l) may add to each opposite
// pair (l, l + 1), and put(l) stores direction l. rho is the reference's
// dd_param. 4- and 8-byte populations are stored as soon as their pair has its
// values: the stores spread over the collision (62^3 FP32 13.5 us a pair of
// steps against 13.8 with all stores at the end, 229 x 186 x 141 with outputs
// 354 against 359). 2-byte ones all at the end (LATE; 512^3 F16S 3.74 ms
// against 3.81): the empty statements that read the results keep the stores
// behind them.
template <bool LATE, class C, class Terms, class Put>
__device__ __forceinline__ void relax(C (&d)[kQ], C rho, C ux, C uy, C uz, C inv_tau, Terms terms,
                                      Put put)
{
    for_pairs(ux, uy, uz, [&](int p, int m, C v, C w) {
        C ep, em;
        equilibrium_pair(ep, em, rho, v, w);
        d[p] += inv_tau * (ep - d[p]);
        d[m] += inv_tau * (em - d[m]);
        terms(p);
        if (!LATE) {
            put(p);
            put(m);
        }
    });
    d[18] += inv_tau * (eq_18(rho) - d[18]);
    if (!LATE) {
        put(18);
        return;
    }
#pragma unroll
    for (int l = 0; l < kQ; l++)
        d[l] = fresh(d[l]);
#pragma unroll
    for (int l = 0; l < kQ; l++)
        put(l);
}

// A VELOCITY_INJECTION cell takes the equilibrium of the lid velocity and
// rho = 1 instead of relaxing: with d = 0 and inv_tau = 1 the relaxation gives
// 0 + 1 * (eq - 0), the equilibrium's own bits. The test is on the whole wave:
// waves without a lid cell pay one scalar branch, not 19 selects or copies.
template <class C>
__device__ __forceinline__ void inject(bool lid_cell, C (&d)[kQ], C& rho, C& ux, C& uy, C& uz,
                                       C& inv_tau, C lid)
{
    if (!__builtin_amdgcn_ballot_w64(lid_cell))
        return;
#pragma unroll
    for (int l = 0; l < kQ; l++)
        d[l] = lid_cell ? (C)0 : d[l];
    inv_tau = lid_cell ? (C)1 : inv_tau;
    ux = lid_cell ? lid : ux;
    uy = lid_cell ? (C)0 : uy;
    uz = lid_cell ? (C)0 : uz;
    rho = lid_cell ? (C)1 : rho;
}

// The gravity terms of alpha (CLbmAlphaCPU.cpp:199-325): the k-th scales the
// one before it (the reference's `tmp` is a #define for `rho`, the first
// scales rho itself), and is added to direction 2 k and subtracted from
// 2 k + 1.
template <class C>
__device__ __forceinline__ C gravity_factor(int k, C g0, C g1, C g2)
{
    switch (k) {
    case 0: return g0 * ((C)1 / (C)18);
    case 1: return g1 * ((C)-1 / (C)18);
    case 2: return (g0 - g1) * ((C)1 / (C)36);
    case 3: return (g0 + g1) * ((C)1 / (C)36);
    case 4: return (g0 + g2) * ((C)1 / (C)36);
    case 5: return (g0 - g2) * ((C)1 / (C)36);
    case 6: return (g2 - g1) * ((C)1 / (C)36);
    case 7: return (g2 + g1) * ((C)-1 / (C)36);
    default: return g2 * ((C)1 / (C)18);
    }
}

// ----------------------------------------------------------------- alpha ---

// One cell of CLbmAlphaCPU::alphaKernelCPU (CLbmAlphaCPU.cpp:75-494). The
// stored density is the last gravity term (add_gravity). `flag` is the cell's
// flag, passed in so a caller that already holds it skips a load.
template <class P, int XF = kXfPack, class A>
__device__ __forceinline__ void alpha_cell(const StepArgs<typename P::C>& a, uint32_t id,
                                           int flag, const A& acc)
{
    using C = typename P::C;
    uint32_t row = 0;
    bool pl = false, pr = false, ul = false, ur = false;
    if (XF != kXfNone)
        xpack_where(a, id, row, pl, pr, ul, ur);
    if (XF != kXfUnpack)
        ul = ur = false;
    const bool pack = pl || pr;
    const bool unpack = ul || ur;
    const int odd = xunpack_odd<0>(ul);
    // The slots are loaded for every cell, whatever its flag, so that the
    // flag's latency overlaps theirs instead of preceding them. GHOST_LAYER
    // (skipped by the reference, :75-76) and OBSTACLE without outputs then
    // store nothing below.
    C d[kQ];
#pragma unroll
    for (int l = 0; l < kQ; l++)
        d[l] = P::load(acc.load(l, 0), l);
    C u[5];
    if (unpack)
        xunpack_load<P, 0>(a, row, ul, odd, u);
    // keeps the flag test (and its wait) below the issued loads
    __builtin_amdgcn_sched_barrier(0);
    if (unpack) {
        uint32_t uov = 0;
        // a cell that stores nothing (GHOST_LAYER, OBSTACLE) leaves the
        // received values where the unpack would have put them: the unpack's
        // codes, encoded from the buffer values (decoding and encoding again
        // need not give them back); written here, so that the received values
        // are not kept across the collision
        const bool keep = flag == kGhostLayer || flag == kObstacle;
#pragma unroll
        for (int k = 0; k < 5; k++) {
            const int e = xplane(k);
            const C v = xunpack_value<P>(u[k], e, uov);
            d[e] = odd ? d[e] : v;
            d[e + 1] = odd ? v : d[e + 1];
            if (keep) {
                if (odd)
                    acc.store(e + 1, 0, P::store(u[k], e));
                else
                    acc.store(e, 0, P::store(u[k], e));
            }
        }
        raise_overflow<P>(a.status, uov);
    }
    if (flag == kGhostLayer) {   // packs its unchanged slots on a send plane
        xpack_alpha<P>(a, row, pl, pr, d);
        return;
    }
    C rho, ux, uy, uz;
    moments(d, rho, ux, uy, uz);

    if (flag == kFluid || flag == kVelocityInjection) {
        C inv_tau = a.inv_tau;
        inject(flag == kVelocityInjection, d, rho, ux, uy, uz, inv_tau, a.lid);
        const C vel2 = ux * ux + uy * uy + uz * uz;
        // direction l goes to slot opp(l) of this cell
        uint32_t ov = 0;
        const A to = acc.for_stores();
        // Without gravity its terms add +-0 to every direction, which changes
        // nothing as long as rho is finite, and leave +-0 as the stored density
        // (rest_rho * rho has its sign); a non-finite rho makes every term NaN,
        // so waves that hold one take them too.
        const bool terms = a.gravity || __builtin_amdgcn_ballot_w64(!__builtin_isfinite(rho));
        C term = rho;
        relax<sizeof(typename P::S) == 2>(
            d, rho - ((C)3 / (C)2) * vel2, ux, uy, uz, inv_tau,
            [&](int l) {
                if (terms) {
                    term = gravity_factor(l / 2, a.g0, a.g1, a.g2) * term;
                    d[l + 1] -= term;
                    d[l] += term;
                }
            },
            [&](int l) { to.store(opp(l), 0, P::store_checked(d[l], opp(l), ov)); });
        rho = terms ? term : a.rest_rho * rho;
        raise_overflow<P>(a.status, ov);
        if (pack) {
            C out[kQ];
#pragma unroll
            for (int s2 = 0; s2 < kQ; s2++)
                out[s2] = d[opp(s2)];
            xpack_alpha<P>(a, row, pl, pr, out);
        }
    } else if (flag == kObstacle) {
        // no stores: the A-A layout makes bounce-back implicit (:330-343)
        if (pack)
            xpack_alpha<P>(a, row, pl, pr, d);
        if (a.store_u) {
            ux = (C)0;
            uy = (C)0;
            uz = (C)0;
        }
    }

    acc.outputs(a, id, rho, ux, uy, uz);
}


// ------------------------------------------------------------------ beta ---

// One cell of CLbmBetaCPU::betaKernelCPU (CLbmBetaCPU.cpp:83-451).
// `dd_param` is a #define for `rho` (:224): the stored FLUID density is
// rho - 1.5 |j|^2. OBSTACLE swaps opposite pairs, which writes back exactly
// what was read, so its stores are skipped. GHOST_LAYER passes values through.
// Neighbour indices wrap modulo the cell count (domainWrap, :44-50). `flag`
// is the cell's flag, as for alpha_cell.
template <class P, int XF = kXfPack, class A>
__device__ __forceinline__ void beta_cell(const StepArgs<typename P::C>& a, uint32_t id,
                                          int flag, const A& acc)
{
    using C = typename P::C;
    uint32_t row = 0;
    bool pl = false, pr = false, ul = false, ur = false;
    if (XF != kXfNone)
        xpack_where(a, id, row, pl, pr, ul, ur);
    if (XF != kXfUnpack)
        ul = ur = false;
    const bool pack = pl || pr;
    const bool unpack = ul || ur;
    const int odd = xunpack_odd<1>(ul);
    // plane l at id + c_l holds direction opp(l) arriving at this cell. As in
    // alpha_cell the slots are loaded whatever the flag (the caller's accessor
    // keeps every neighbour index in bounds); OBSTACLE, which writes back what
    // it reads, stores nothing below.
    C d[kQ];
#pragma unroll
    for (int l = 0; l < kQ; l++)
        d[opp(l)] = P::load(acc.load(l, cx(l) + cy(l) * a.nx + cz(l) * a.nxy), l);
    C u[5];
    if (unpack)
        xunpack_load<P, 1>(a, row, ul, odd, u);
    __builtin_amdgcn_sched_barrier(0);
    if (unpack) {
        // slot l's value is d[opp(l)]: slot e in d[e + 1], slot e + 1 in d[e].
        // OBSTACLE stores nothing: the received values stay where the unpack
        // puts them (written here, so they are not kept across the collision)
        uint32_t uov = 0;
        const bool keep = flag == kObstacle;
#pragma unroll
        for (int k = 0; k < 5; k++) {
            const int e = xplane(k);
            const C v = xunpack_value<P>(u[k], e, uov);
            d[e + 1] = odd ? d[e + 1] : v;
            d[e] = odd ? v : d[e];
            if (keep) {
                if (odd)
                    acc.store(e + 1, cx(e + 1) + cy(e + 1) * a.nx + cz(e + 1) * a.nxy,
                              P::store(u[k], e));
                else
                    acc.store(e, cx(e) + cy(e) * a.nx + cz(e) * a.nxy, P::store(u[k], e));
            }
        }
        raise_overflow<P>(a.status, uov);
    }

    C rho, ux, uy, uz;
    moments(d, rho, ux, uy, uz);

    // direction l goes to slot l of neighbour id + c_l
    uint32_t ov = 0;
    auto put = [&](const A& to, int l) {
        to.store(l, cx(l) + cy(l) * a.nx + cz(l) * a.nxy, P::store_checked(d[l], l, ov));
    };
    // The collision comes last: a branch after it that still read the arriving
    // values would keep all 19 in registers of their own (FP32 64 VGPRs instead
    // of 40, FP64 118 instead of 70). `kind` goes through an empty statement so
    // that the branches stay in this order.
    constexpr int kStill = 0, kPass = 1, kMoving = 2;
    const int kind = fresh(flag == kFluid || flag == kVelocityInjection ? kMoving
                           : flag == kObstacle                          ? kStill
                                                                        : kPass);
    if (kind == kStill) {
        if (pack) {
            // the swap writes back the value read from plane l (:302-311)
            C out[kQ];
#pragma unroll
            for (int l = 0; l < kQ; l++)
                out[l] = d[opp(l)];
            xpack_beta<P>(a, row, pl, pr, out);
        }
        if (a.store_u) {
            ux = (C)0;
            uy = (C)0;
            uz = (C)0;
        }
    }
    if (kind == kPass) {
        const A to = acc.for_stores();
#pragma unroll
        for (int l = 0; l < kQ; l++)
            put(to, l);
    }
    if (kind == kMoving) {
        C inv_tau = a.inv_tau;
        inject(flag == kVelocityInjection, d, rho, ux, uy, uz, inv_tau, a.lid);
        const C vel2 = ux * ux + uy * uy + uz * uz;
        rho = rho - ((C)3 / (C)2) * (vel2);
        const A to = acc.for_stores();
        relax<sizeof(typename P::S) == 2>(d, rho, ux, uy, uz, inv_tau, [](int) {},
                                          [&](int l) { put(to, l); });
    }
    raise_overflow<P>(a.status, ov);
    if (pack && kind != kStill)
        xpack_beta<P>(a, row, pl, pr, d);

    acc.outputs(a, id, rho, ux, uy, uz);
}

// ------------------------------------------------ two cells per thread ---

// A cell's rho and u on their way to the pair's stores; GHOST_LAYER cells give
// none in alpha.
struct HalfOutputs {
    float rho, u[3];
    bool given = false;
};

// Two neighbouring cells per thread for the 16-bit formats: every access moves
// both cells' codes of a plane in one 4-byte word (beta's planes start at any
// even byte; unaligned words cost the memory nothing more than the shifted
// halves did). The cells take the per-cell code in turn, reading and writing
// their halves of the words in registers. A cell that stores nothing keeps what a
// face transfer on another stream puts into its slots meanwhile: beside it the
// other cell stores its halves alone. GHOST_LAYER cells in alpha are such cells,
// and OBSTACLE cells too where a face of the domain is exchanged (a GHOST_LAYER
// face). The walls of a closed domain are stored back as they were read
// (store_walls): without them no row's first and last lines are whole, and the
// memory then reads what it writes (512^3 F16S 3925 us for an alpha and a beta
// against 3740, 250^3 462 against 421; with nontemporal stores 4360 and 519).
// Bound by memory: F16S 512^3 moves its 20.8 GB of an alpha and a beta in 3740 to
// 3880 us by the allocation, 5.4 to 5.6 TB/s (one cell per thread 4050 to 4180).
template <class S>
struct AccHalf {
    uint32_t* word;   // [19], registers
    HalfOutputs* out;
    int high;
    __device__ __forceinline__ void outputs(const StepArgs<float>&, uint32_t, float rho, float ux,
                                            float uy, float uz) const
    {
        *out = HalfOutputs{rho, {ux, uy, uz}, true};
    }
    __device__ __forceinline__ AccHalf for_stores() const { return *this; }
    __device__ __forceinline__ S load(int l, int32_t) const
    {
        return __builtin_bit_cast(S, (uint16_t)(high ? word[l] >> 16 : word[l]));
    }
    __device__ __forceinline__ void store(int l, int32_t, S v) const
    {
        const uint32_t c = __builtin_bit_cast(uint16_t, v);
        word[l] = high ? (word[l] & 0xFFFFu) | (c << 16) : (word[l] & 0xFFFF0000u) | c;
    }
};

using Word16 = uint32_t __attribute__((aligned(2)));

template <bool NT>
__device__ __forceinline__ uint32_t load_word(const char* base, uint32_t off)
{
    const LBM_GLOBAL Word16* p = (const LBM_GLOBAL Word16*)(base + off);
    return NT ? __builtin_nontemporal_load(p) : *p;
}
template <bool NT, class T, class V>
__device__ __forceinline__ void store_at(const char* base, uint32_t off, V v)
{
    LBM_GLOBAL T* p = (LBM_GLOBAL T*)(const_cast<char*>(base) + off);
    if (NT)
        __builtin_nontemporal_store((T)v, p);
    else
        *p = (T)v;
}

// The words of the cells that store: both halves, or one (never nontemporal: its
// line is its neighbours' too).
template <bool NT>
__device__ __forceinline__ void store_cells(const char* const* plane, uint32_t off,
                                            const uint32_t (&w)[kQ], bool low, bool high)
{
    if (low && high) {
#pragma unroll
        for (int l = 0; l < kQ; l++)
            store_at<NT, Word16>(plane[l], off, w[l]);
    } else if (low || high) {
        const uint32_t at = off + (high ? 2 : 0), shift = high ? 16 : 0;
#pragma unroll
        for (int l = 0; l < kQ; l++)
            store_at<false, uint16_t>(plane[l], at, w[l] >> shift);
    }
}

// Both cells' rho and u, 8 bytes at a time (id is even and the fields' planes
// are multiples of 256 elements apart).
__device__ __forceinline__ void store_outputs(const StepArgs<float>& a, uint32_t id,
                                              const HalfOutputs (&o)[2])
{
    if (!a.store_u && !a.store_rho)
        return;
    if (o[0].given && o[1].given) {
        if (a.store_u)
#pragma unroll
            for (int k = 0; k < 3; k++)
                *(float2*)(a.u + k * a.stride + id) = make_float2(o[0].u[k], o[1].u[k]);
        if (a.store_rho)
            *(float2*)(a.rho + id) = make_float2(o[0].rho, o[1].rho);
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (o[h].given)
            CellOutputs().outputs(a, id + h, o[h].rho, o[h].u[0], o[h].u[1], o[h].u[2]);
}

// Cells id and id + 1 of alpha (id even; the last cell of an odd number alone).
template <class P, bool NT>
__device__ __forceinline__ void alpha_pair(const StepArgs<typename P::C>& a, uint32_t id)
{
    using S = typename P::S;
    const LBM_GLOBAL uint8_t* fp = (const LBM_GLOBAL uint8_t*)a.flags + id;
    const uint32_t off = id * (uint32_t)sizeof(S);
    if (id + 1 >= (uint32_t)a.n) {
        if (id < (uint32_t)a.n)
            alpha_cell<P, kXfNone>(a, id, *fp, Acc32<S, NT>{a.plane, off});
        return;
    }
    uint32_t w[kQ];
    const uint32_t flags = *(const LBM_GLOBAL uint16_t*)fp;
#pragma unroll
    for (int l = 0; l < kQ; l++)
        w[l] = load_word<NT>(a.plane[l], off);
    const int f0 = flags & 255, f1 = flags >> 8;
    HalfOutputs o[2];
    alpha_cell<P, kXfNone>(a, id, f0, AccHalf<S>{w, &o[0], 0});
    alpha_cell<P, kXfNone>(a, id + 1, f1, AccHalf<S>{w, &o[1], 1});
    store_outputs(a, id, o);
    auto moves = [](int f) { return f == kFluid || f == kVelocityInjection; };
    auto stores = [&](int f) { return moves(f) || (f == kObstacle && a.store_walls); };
    if (moves(f0) || moves(f1))
        store_cells<NT>(a.plane, fresh(off), w, stores(f0), stores(f1));
}

// Cells id and id + 1 (id even) of beta, none of whose neighbours wrap.
template <class P>
__device__ __forceinline__ void beta_pair(const StepArgs<typename P::C>& a, uint32_t id)
{
    using S = typename P::S;
    const uint32_t off = id * (uint32_t)sizeof(S);
    uint32_t w[kQ];
    const uint32_t flags = *(const LBM_GLOBAL uint16_t*)((const LBM_GLOBAL uint8_t*)a.flags + id);
#pragma unroll
    for (int l = 0; l < kQ; l++)
        w[l] = load_word<false>(a.plane[l], off);
    const int f0 = flags & 255, f1 = flags >> 8;
    HalfOutputs o[2];
    beta_cell<P, kXfNone>(a, id, f0, AccHalf<S>{w, &o[0], 0});
    beta_cell<P, kXfNone>(a, id + 1, f1, AccHalf<S>{w, &o[1], 1});
    store_outputs(a, id, o);
    auto stores = [&](int f) { return f != kObstacle || a.store_walls; };
    if (f0 != kObstacle || f1 != kObstacle)
        store_cells<false>(a.plane, fresh(off), w, stores(f0), stores(f1));
}


}  // namespace lbm
