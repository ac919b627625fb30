// Internal declarations of the HIP solver (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <limits>
#include <string>

#include "lbm_abi.h"

namespace lbm {

// Unsigned 32-bit division by a runtime constant: q = (umulhi(n, m) + n) >> s,
// exact for every 32-bit n (round-up multiplier, Granlund & Montgomery 1994).
struct FastDiv {
    uint32_t d = 1, m = 0, s = 0;
    FastDiv() = default;
    explicit FastDiv(uint32_t div) : d(div)
    {
        uint32_t l = 0;
        while (l < 32 && (1ull << l) < div)
            l++;
        s = l;
        m = (uint32_t)((((1ull << l) - div) << 32) / div + 1);
        if (div == 1)
            m = 0, s = 0;
    }
    __device__ __forceinline__ uint32_t div(uint32_t n) const
    {
        return (uint32_t)(((uint64_t)__umulhi(n, m) + n) >> s);
    }
};

// A box of cells in halo coordinates.
struct Box {
    int ox, oy, oz;
    int bx, by, bz;
    uint32_t cells() const { return (uint32_t)bx * (uint32_t)by * (uint32_t)bz; }
};

// Everything a step kernel needs, passed by value.
template <class C>
struct StepArgs {
    void* dd;
    const uint8_t* flags;
    C* rho;
    C* u;
    int64_t stride;   // elements between planes
    int32_t n;        // cells with halo
    int32_t nx, nxy;  // row and slab strides
    int32_t ox, oy, oz;
    uint32_t cells;   // cells of the box
    FastDiv div_bx, div_by;
    C inv_tau, lid, g0, g1, g2;
    int gravity;      // any of g0, g1, g2 is not zero
    C rest_rho;       // gravity_product, used when g is zero
    int store_rho, store_u;
    int xcd;          // renumber workgroups per XCD
    int reverse;      // workgroups take the blocks of cells from the last to the first
    // byte address of plane l, shifted by the neighbour offset of direction l
    // for beta (0 for alpha): uniform per-plane bases for 32-bit lane offsets
    const char* plane[19];
    // fused x-face pack: dense face buffers [slot][z * ny + y] (LEFT, RIGHT)
    C* xpack[2];
    // fused x-face unpack: the received face buffers, same layout (LEFT, RIGHT)
    const C* xunpack[2];
    int xpack_on;     // any of xpack / xunpack set
    FastDiv div_nx;
    int32_t ny;
    int32_t fcells;   // ny * nz
    // set to 1 by a store the storage format cannot represent (F16C)
    uint32_t* status;
    // 16-bit pairs may store OBSTACLE cells back (is_closed). Kept last: among
    // the fields above it moved the pointers' alignment, and small domains took
    // 3 to 5 % longer (30^3 FP32 7.5 us for an alpha and a beta against 7.1).
    int store_walls;
};

// What alpha's gravity terms multiply rho by in all (CLbmAlphaCPU.cpp:199-325,
// without the weights, whose two signs cancel). With g = 0: +-0, the sign of
// the stored density.
template <class C>
inline C gravity_product(C g0, C g1, C g2)
{
    return ((g0 * g1 * (g0 - g1)) * ((g0 + g1) * (g0 + g2) * (g0 - g2))) *
           ((g2 - g1) * (g2 + g1) * g2);
}
inline int has_gravity(const double (&g)[3]) { return g[0] != 0 || g[1] != 0 || g[2] != 0; }

}  // namespace lbm

struct lbm_solver {
    lbm_params p;
    int size_h[3];
    int64_t n;         // cells with halo
    int64_t stride;    // plane stride in elements
    int elem_bytes;    // bytes per stored population
    int out_bytes;     // bytes per rho/u element (4 or 8)
    void* dd;
    uint8_t* flags;
    void* rho;
    void* u;
    void* staging;     // device staging for host copies
    size_t staging_bytes;
    double* partials;  // reduction partials (kReduceBlocks * 5) followed by 5 results
    double* result;    // pinned host memory for 5 results, NULL when none was free
    void* residual_prev;  // momentum saved by lbm_residual, 3 planes of the compute type
    int residual_valid;
    int launch[2];     // LBM_LAUNCH_* options of the alpha and beta kernels
    int launch_set[2]; // set by the caller: kept when the step pack changes
    void* xpack[2];    // fused x-face pack buffers (LEFT, RIGHT), NULL when off
    const void* xunpack[2];  // fused x-face unpack buffers (LEFT, RIGHT), NULL when off
    void* dd_alt;      // second population buffer of the out-of-place pair pass
    uint32_t* status;  // device word: nonzero after a store out of the storage range
    // the device's counter of stepped bytes (lbm_abi.cpp) at this solver's last
    // half-step, the bytes of other solvers before that one, its kernel (-1: the
    // state was written since) and whether its stores were nontemporal
    uint64_t step_mark, step_gap;
    int last_kernel, streamed;
};

namespace lbm {

void set_error(const std::string& msg);
int hip_fail(hipError_t e, const char* what);

hipError_t launch_init(const lbm_solver* s, hipStream_t st, int write_flags);
hipError_t launch_alpha(const lbm_solver* s, const Box& b, int opts, hipStream_t st);
hipError_t launch_beta(const lbm_solver* s, const Box& b, int opts, hipStream_t st);

// field: 0 populations (the lattice vectors of `mask`; buffers keep all 19
// planes), 1 velocities (3), 2 densities (1)
hipError_t launch_box_get(const lbm_solver* s, int field, const Box& b, void* dst,
                          uint32_t mask, hipStream_t st);
// the population copies of two boxes (the faces of one axis) in one launch,
// each with its own buffer and plane mask
hipError_t launch_dd_get_pair(const lbm_solver* s, const Box* b, void* const* dst,
                              const uint32_t* mask, hipStream_t st);
// faces of one solver copied into another's with no buffer
// (lbm_exchange_face[s]): the boxes of a transfer have the same extents, the
// solvers one device and precision, and no element is written by one
// transfer of the list and read or written by another
struct XferDesc {
    const lbm_solver* from;
    Box sb;
    lbm_solver* to;
    Box db;
    uint32_t mask;
};
constexpr int kXferBatch = 8;   // transfers per launch
hipError_t launch_dd_xfer(const XferDesc* list, int n, hipStream_t st);
hipError_t launch_dd_set_pair(const lbm_solver* s, const Box* b, const void* const* src,
                              const uint32_t* mask, hipStream_t st);
// both x faces in one launch (nt: streaming stores)
hipError_t launch_set_dd_xpair(const lbm_solver* s, const void* lo, const void* hi, int x_lo,
                               int x_hi, uint32_t mask_lo, uint32_t mask_hi, bool nt,
                               hipStream_t st);
hipError_t launch_box_set(const lbm_solver* s, int field, const Box& b, const void* src,
                          uint32_t mask, hipStream_t st);
hipError_t launch_flags_get(const lbm_solver* s, const Box& b, int32_t* dst, hipStream_t st);
hipError_t launch_flags_set(const lbm_solver* s, const Box& b, const int32_t* src,
                            hipStream_t st);

hipError_t launch_reduce_box(const lbm_solver* s, const Box& b, double* partials,
                             double* out_dev, hipStream_t st);
hipError_t launch_moments(const lbm_solver* s, const Box& b, int layout, void* dst,
                          hipStream_t st);
hipError_t launch_residual(const lbm_solver* s, int layout, double* partials, double* out_dev,
                           hipStream_t st);
// One solver's residual inputs, for the residual of many solvers in one launch
// (partials: count * kReduceBlocks * 5 doubles; out: count * 5).
struct ResidualMember {
    const void* dd;
    const uint8_t* flags;
    void* prev;
    int64_t stride;
    uint32_t n;
    const uint32_t* status;
};
hipError_t launch_residual_members(int precision, const ResidualMember* mem, int count,
                                   int layout, double* partials, double* out_dev,
                                   hipStream_t st);

constexpr int kReduceBlocks = 1024;   // at most: 4 workgroups on each of 256 CUs
// Per-solver reduction buffer: kReduceBlocks * 5 partial sums, 5 results,
// then the solver's overflow word (lbm_solver::status).
constexpr size_t kPartialsBytes = (size_t)(kReduceBlocks + 1) * 5 * sizeof(double) + 64;

// lbm_reduce_boxes_noalloc: the device address of the static partials array
// on `device` (which must be current), looked up on the first call per device.
hipError_t noalloc_scratch(int device, double** ptr);
// k_reduce_box for count (<= LBM_NOALLOC_MAX_BOXES) boxes of solvers of one
// precision; partials: count * kReduceBlocks * 5 doubles, out: count * 5.
hipError_t launch_reduce_boxes(const lbm_solver* const* s, const Box* b, int count,
                               double* partials, double* out_dev, hipStream_t st);

// Default launch options of the step kernels (kernel 0 = alpha, 1 = beta),
// measured on MI355X: FP32 and FP64 gain from fewer resident waves (fewer
// concurrent plane streams), 16-bit storage needs every wave; F64 beta from
// line-aligned accesses staged through LDS. FP32 from 512-thread workgroups
// of two cells per thread on large domains (wide: at 192^3 and up; below
// about 160^3 they leave too few workgroups); with the fused x-face pack
// (with_pack) FP32 beta on large domains runs in 1024-thread workgroups, one
// per CU, and FP32 alpha on small domains keeps 3 waves per SIMD (measured
// with the six-face exchange at 512^3). 16-bit storage: cached
// accesses; F16S and BF16S beta in 1024-thread workgroups on large domains
// (F16C beta, with more integer work per cell, loses with them).
constexpr int64_t kWideCells = 6 << 20;   // halo-inclusive cells for `wide`

// 32-bit byte offsets reach every element of a plane
inline bool plane_off32(const lbm_solver* s)
{
    return (uint64_t)s->stride * (uint64_t)s->elem_bytes < (1ull << 32);
}

// addr64: the planes need 64-bit element offsets (4 GiB and up); the FP32
// beta with the fused unpack keeps 512-thread workgroups there, chosen when
// the 1024-thread kernel spilled (it needs 85 of its 128 registers now).
inline int default_launch(int precision, int kernel, bool with_pack, bool wide,
                          bool with_unpack = false, bool addr64 = false)
{
    switch (precision) {
    case LBM_F32:
        if (kernel == 0) {
            // 256-thread workgroups, 3 waves per SIMD: with a step pack on a
            // small domain, and with the fused x-face unpack (whose received
            // loads hold a wave longer than the streaming 2-wave shape allows)
            if (with_unpack || (with_pack && !wide))
                return LBM_LAUNCH_NONTEMPORAL | LBM_LAUNCH_WAVES3;
            return (wide ? LBM_LAUNCH_WIDE : 0) | LBM_LAUNCH_NONTEMPORAL | LBM_LAUNCH_WAVES2;
        }
        if (with_unpack && wide && addr64)
            return LBM_LAUNCH_WIDE | LBM_LAUNCH_WAVES3;
        if ((with_pack || with_unpack) && wide)
            return LBM_LAUNCH_BIG | LBM_LAUNCH_WAVES4;
        return (wide ? LBM_LAUNCH_WIDE : 0) | LBM_LAUNCH_WAVES2;
    case LBM_F64:
        return kernel == 0 ? (LBM_LAUNCH_NONTEMPORAL | LBM_LAUNCH_WAVES2)
                           : (LBM_LAUNCH_LDS | LBM_LAUNCH_WAVES2);
    case LBM_F16C:
        return 0;
    default:
        // 1024-thread beta workgroups wait on their slowest wave: with the
        // fused unpack's received loads 256-thread ones are faster
        return kernel == 1 && wide && !with_unpack ? LBM_LAUNCH_BIG : 0;
    }
}

inline bool is_full(const lbm_solver* s, const Box& b)
{
    return b.ox == 0 && b.oy == 0 && b.oz == 0 && b.bx == s->size_h[0] &&
           b.by == s->size_h[1] && b.bz == s->size_h[2];
}

// No face of the domain was created to be exchanged.
inline bool is_closed(const lbm_solver* s)
{
    for (int face : s->p.bc)
        if (face == LBM_GHOST_LAYER)
            return false;
    return true;
}

// Bytes a half-step of the whole domain reads and writes in place.
inline uint64_t resident_bytes(const lbm_solver* s)
{
    const uint64_t out = (s->p.store_densities ? 1 : 0) + (s->p.store_velocities ? 3 : 0);
    return (uint64_t)s->n * (19 * s->elem_bytes + 1 + out * s->out_bytes);
}

// Domains up to here keep plain launches (options_of_step).
constexpr uint64_t kTinyBytes = 2ull << 20;

// Internal launch options beside the LBM_LAUNCH_* ones.
constexpr int kPairCells = 1 << 16;   // 16-bit formats: two neighbouring cells per thread
constexpr int kReverse = 1 << 17;     // the last cells first

// Launch options of a whole-domain step without face work whose kernel the
// caller has not set. What decides is whether the state still lies in a cache
// when the step starts: near and far are the lesser and the greater of the
// bytes of other solvers stepped between this half-step and the solver's last,
// and between that one and its predecessor. Times are us for an alpha and a
// beta; "in turn": three solvers, one alpha and beta each. The same launches in
// another allocation differ by 1 to 3 %, in another process by up to 10: both
// sides of a line were timed in one process, in several allocations.
//  * Own bytes up to about the 8 L2s (4 MiB each): every workgroup is resident
//    at once and no cap on the waves pays (62^3 FP32, 19 MB: 13.4 against 15.9
//    with the streaming options). Both steps give each XCD the same contiguous
//    range of cells, so that its L2 still holds them, and the z neighbours of
//    beta, from one half-step to the next: 24 x 90 x 90 FP32 13.2 against 17.7
//    without the map, 75^3 20.4 / 23.5, 50^3 FP64 16.3 / 21.3, 75^3 F16S 17.1 /
//    20.3. Slabs of a multiple of 8 workgroups, whose z neighbours lie on one XCD
//    by themselves, gain too (FP32 3 % on average over 12 extents, 254 x 6 x 98
//    10.8 / 14.1). FP32 and FP64 planes a multiple of 512 KiB apart share sets
//    of the L2s, by the allocation: 62^3 FP32 12.1 or 14.3 against 13.4, with rho
//    and u 13.5 or 15.6 / 14.1, on average over 7 such extents the same. Not
//    below kTinyBytes (16^3 7.1 against 6.7).
//  * All within the 256 MB Infinity Cache (one cavity stepped again and again):
//    alpha cached and uncapped, beta with one contiguous range of cells per
//    XCD, whose L2 then serves the lines that neighbouring workgroups share:
//    104^3 FP32 57.5 against 67-74, 140^3 129 against 147-150, FP64 112^3 134
//    against 163.
//  * Only the state itself fits (a few steps, then another solver's turn): the
//    XCD map loses for FP32 and FP64; beta in 1024-thread workgroups (FP32
//    120^3 95.0 against 98.8 in 256-thread ones, 140^3 142.6 against 147.6),
//    FP64 at 3 waves per SIMD (110^3 140.7 against 146.9); F16S with the map
//    (150^3 88.0 against 93.1), F16C without (two 180^3 158 against 175).
//  * The state does not fit: beta takes the cells from the last to the first
//    (kReverse), alpha from the first. Each then starts with what the other
//    has just left in the Infinity Cache, up to 250 MB that need not come from
//    HBM, as long as alpha stores them there (no nontemporal alpha). 185^3 FP32
//    320 against 351, in turn 340 against 385; 214^3 512 / 550, 529 / 570; FP64
//    150^3 352 / 384, 377 / 414, 200^3 930 / 923, 972 / 967. Alpha at 2 waves per
//    SIMD; FP32 up to 600 MB with nothing else between at 4 (163^3 224 against
//    232, 185^3 320 / 330, 214^3 512 / 512; in turn 4 lose, 214^3 543 against
//    530). Beta FP32 in 1024-thread workgroups, from 1.6 GB through LDS (235^3
//    701 against 720, 270^3 1088 / 1087, 340^3 2217 / 2193, 420^3 4240 / 4150),
//    FP64 through LDS from 1.8 GB (225^3 1259 against 1280, 249^3 1790 / 1767,
//    330^3 4340 / 4130). From 3 GB alpha is nontemporal: what it leaves in the
//    cache is little against the rest (FP64 270^3 2217 cached against 2298,
//    290^3 2807 / 2795, 330^3 4130 / 4092; FP32 in turn 340^3 2206 / 2250, 512^3
//    7600 / 7490).
//  * Solvers that fit each but not together, stepped forwards by alpha and
//    backwards by beta (the two gaps differ): the same, beta's range per XCD
//    backwards; eight 82^3 FP32 322 against 344, eight 130^3 1147 against
//    1174, four 162 x 82 x 82 FP64 494 against 521. Stepped round and round,
//    nothing is left of them: nontemporal alpha, no reversal. Nor is after such
//    an alpha (`streamed`), whatever comes between: the first alpha of eight
//    new 128^3 streams, and their first beta backwards with the map took 680
//    with the exchange of the faces, 620 plainly.
//  * The 16-bit formats beyond the L2s take two neighbouring cells per thread
//    (4-byte accesses): F16S 130^3 57.7 against 59.7 for one cell per thread,
//    61 against 64 with others in turn; streaming, 256^3 450 against 505,
//    F16C 512^3 3850 against 4060, BF16S 400^3 1769 against 1893. Within the
//    L2s half the waves lose (62^3 13.2 against 12.4). Their alpha is
//    nontemporal where nothing else comes between (F16S 200^3 211 against 225
//    for a cached one with the reversal, 250^3 421 / 440; from 1.2 GB with the
//    reversal, 400^3 1810 / 1840, F16C 512^3 3440 at 4 waves per SIMD and 3540
//    at 3) and cached with the reversal in turn (200^3 235 against 245, 221^3
//    309 / 340, 270^3 557 / 560) and with rho and u stored below 1.2 GB (221^3
//    356 / 385, 270^3 661 / 724). Domains with GHOST_LAYER faces store half words
//    at their walls and ghosts, which nontemporal neighbours in the line turn
//    into reads of the memory: always cached (250^3 462 against 519, 400^3 1890
//    / 2130).
inline int step_options(const lbm_solver* s, int kernel, uint64_t near, uint64_t far,
                        bool streamed)
{
    constexpr uint64_t MB = 1ull << 20, kL2 = 40 * MB, kCache = 250 * MB;
    constexpr int NT = LBM_LAUNCH_NONTEMPORAL, XCD = LBM_LAUNCH_XCD_REMAP;
    constexpr int W2 = LBM_LAUNCH_WAVES2, W3 = LBM_LAUNCH_WAVES3, W4 = LBM_LAUNCH_WAVES4;
    constexpr int LDS = LBM_LAUNCH_LDS, BIG = LBM_LAUNCH_BIG, REV = kReverse;
    const uint64_t own = resident_bytes(s);
    const int p = s->p.precision;
    if (own <= kL2)
        return XCD;
    if (streamed && own <= kCache)   // the last half-step left nothing in the cache
        near = far = kCache;
    near += own;
    far += own;
    const bool alone = far <= own + own / 4;      // no other solvers in between
    const bool to_and_fro = far >= near + own / 2;
    auto opts = [&](int alpha, int beta) { return kernel == 0 ? alpha : beta; };
    if (p != LBM_F32 && p != LBM_F64) {
        const bool open = !is_closed(s), large = own > 1200 * MB;
        const bool outputs = s->p.store_densities || s->p.store_velocities;
        int o;
        if (near <= kCache)
            o = far <= 300 * MB ? opts(0, XCD | W4) : p == LBM_F16C ? W4 : opts(W4, XCD | W3);
        else if (own <= kCache)
            o = opts(open ? W3 : NT | W3, XCD | W4);
        else if (open || (!large && (outputs || !alone)))
            o = opts(W3, W4 | REV);
        else if (!large)
            o = opts(NT | W4, W4);
        else   // F16C has more integer work per cell
            o = p == LBM_F16C ? opts(NT | W4, W4 | REV) : opts(NT | W3, W3 | REV);
        return kPairCells | o;
    }
    if (near <= kCache && far <= 300 * MB)
        return opts(0, XCD | (p == LBM_F32 ? W2 : W3));
    if (near <= kCache)
        return p == LBM_F32 ? opts(W3, BIG | W4) : opts(W2, W3);
    if (own <= kCache)
        return to_and_fro ? opts(W2, XCD | W3 | REV) : opts(NT | W2, W2);
    const int huge = own < 3000 * MB ? 0 : NT;
    if (p == LBM_F32)
        return own >= 1600 * MB ? opts(huge | W2, LDS | W4 | REV)
                                : opts(alone && own <= 600 * MB ? W4 : W2, BIG | W4 | REV);
    return opts(huge | W2, (own < 1800 * MB ? 0 : LDS) | W2 | REV);
}

// ||u - u_prev|| / ||u|| from the two FP64 sums; a non-finite state gives NaN
// (never a small number that would pass a convergence test).
inline double residual_ratio(double num, double den)
{
    if (std::isnan(num) || std::isnan(den) || std::isinf(num) || std::isinf(den))
        return std::numeric_limits<double>::quiet_NaN();
    if (den > 0)
        return std::sqrt(num / den);
    return num > 0 ? std::numeric_limits<double>::infinity() : 0.0;
}

// The residual call's value: residual_ratio, except on the first call after
// creation, reset or load, where no previous field exists (num compares with
// a stale snapshot): +inf, or NaN when the current field (den) is already
// non-finite.
inline double first_residual(int valid, double num, double den)
{
    if (valid)
        return residual_ratio(num, den);
    if (std::isnan(den) || std::isinf(den))
        return std::numeric_limits<double>::quiet_NaN();
    return std::numeric_limits<double>::infinity();
}

}  // namespace lbm
