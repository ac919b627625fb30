// Host build of the two-cells-per-thread code of the 16-bit steps (lbm_cell.hpp):
// while a pair of cells is stepped, another writer puts new codes into the slots
// of the cell that stores nothing. They have to be there afterwards, and the
// cell that moves has to hold what it gets alone; only OBSTACLE cells of a closed
// domain may be stored back. Prints the number of cases; returns 1 at the first
// that fails.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <vector>

#undef __device__
#undef __host__
#undef __forceinline__
#define __device__
#define __host__
#define __forceinline__ inline
#define __uint_as_float(x) __builtin_bit_cast(float, (uint32_t)(x))
#define __float_as_uint(x) __builtin_bit_cast(uint32_t, (float)(x))
#define __umulhi(a, b) ((uint32_t)(((uint64_t)(a) * (b)) >> 32))
#define __builtin_amdgcn_ballot_w64(x) ((uint64_t)(x))
#define __builtin_amdgcn_sched_barrier(x)
#define __hip_atomic_fetch_or(p, v, order, scope) (*(p) |= (v))
struct {
    uint32_t x;
} blockIdx, gridDim;
// the empty statements of the kernels name vector registers of the GPU
#define asm
#define volatile(...)
#include "lbm_cell.hpp"
#undef asm
#undef volatile

using namespace lbm;

static void (*g_other_writer)() = nullptr;

// The storage format, with the other writer at work at every store.
template <class P>
struct Watched : P {
    static typename P::S store_checked(typename P::C v, int l, uint32_t& ov)
    {
        g_other_writer();
        return P::store_checked(v, l, ov);
    }
};

constexpr int kN = 6, kCells = kN * kN * kN;
static std::vector<uint16_t> g_state;
static std::vector<uint8_t> g_flags;
static int g_phase;
static std::vector<int> g_still;   // cells that store nothing

static size_t slot(int l, int cell)
{
    const int delta = g_phase ? cx(l) + cy(l) * kN + cz(l) * kN * kN : 0;
    return (size_t)l * kCells + cell + delta;
}
static uint16_t received(int l, int cell) { return (uint16_t)(0x1100 + 64 * (cell & 1) + l); }
static void write_still()
{
    for (int c : g_still)
        for (int l = 0; l < kQ; l++)
            g_state[slot(l, c)] = received(l, c);
}

static StepArgs<float> args(bool closed, uint32_t* status)
{
    StepArgs<float> a{};
    a.dd = g_state.data();
    a.flags = g_flags.data();
    a.stride = kCells;
    a.n = kCells;
    a.nx = kN;
    a.nxy = kN * kN;
    a.cells = kCells;
    a.inv_tau = 1.3f;
    a.lid = 0.07f;
    a.store_walls = closed;
    a.status = status;
    for (int l = 0; l < kQ; l++)
        a.plane[l] = (const char*)(g_state.data() + slot(l, 0));
    return a;
}

template <class P>
static bool run(const char* name, bool closed, int* cases)
{
    using S = typename P::S;
    using W = Watched<P>;
    const int id = kN * kN * 2 + kN * 2 + 2;   // even, away from the ends
    const int kinds[4] = {kObstacle, kFluid, kVelocityInjection, kGhostLayer};
    for (g_phase = 0; g_phase < 2; g_phase++)
        for (int f0 : kinds)
            for (int f1 : kinds) {
                std::vector<uint16_t> start(kQ * kCells);
                for (size_t i = 0; i < start.size(); i++)
                    start[i] = __builtin_bit_cast(
                        uint16_t, P::store(weight<float>((int)(i / kCells)) *
                                               (1.0f + 0.01f * (float)((i * 37) % 11)),
                                           (int)(i / kCells)));
                g_flags.assign(kCells, kFluid);
                g_flags[id] = (uint8_t)f0;
                g_flags[id + 1] = (uint8_t)f1;
                auto stores = [&](int f) {
                    return g_phase ? f != kObstacle : f == kFluid || f == kVelocityInjection;
                };
                uint32_t status = 0;
                // each cell alone, nobody else writing
                g_state = start;
                g_still.clear();
                g_other_writer = [] {};
                for (int c = id; c < id + 2; c++) {
                    const auto a = args(closed, &status);
                    const Acc32<S, false> acc{a.plane, (uint32_t)(c * sizeof(S))};
                    if (g_phase)
                        beta_cell<W, kXfNone>(a, c, g_flags[c], acc);
                    else
                        alpha_cell<W, kXfNone>(a, c, g_flags[c], acc);
                }
                std::vector<uint16_t> want = g_state;
                // the pair, with the other writer
                g_state = start;
                for (int c = id; c < id + 2; c++)
                    if (!stores(g_flags[c]))
                        g_still.push_back(c);
                g_other_writer = write_still;
                const auto a = args(closed, &status);
                if (g_phase)
                    beta_pair<W>(a, id);
                else
                    alpha_pair<W, false>(a, id);
                if (g_still.size() < 2)
                    for (int c : g_still)
                        for (int l = 0; l < kQ; l++)
                            want[slot(l, c)] = closed && g_flags[c] == kObstacle
                                                   ? g_state[slot(l, c)]
                                                   : received(l, c);
                (*cases)++;
                if (g_state != want) {
                    size_t i = 0;
                    while (g_state[i] == want[i])
                        i++;
                    printf("%s %s %s, flags %d %d: plane %d cell %d is %04x, not %04x\n", name,
                           closed ? "closed" : "open", g_phase ? "beta" : "alpha", f0, f1, (int)(i / kCells),
                           (int)(i % kCells) - id, g_state[i], want[i]);
                    return false;
                }
            }
    return true;
}

int main()
{
    int cases = 0;
    bool ok = true;
    for (bool closed : {false, true})
        ok = ok && run<StoreF16S>("f16s", closed, &cases) &&
             run<StoreBF16S>("bf16s", closed, &cases) && run<StoreF16C>("f16c", closed, &cases);
    printf("%d cases\n", cases);
    return ok ? 0 : 1;
}
