// The launch options that whole-domain steps choose (step_options), for the rows on
// standard input: precision nx ny nz (interior) outputs face near far streamed, one
// line of "alpha beta" for each; near and far are the MiB of other solvers in between.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

#include <iostream>

#undef __device__
#undef __host__
#undef __forceinline__
#define __device__
#define __host__
#define __forceinline__ inline
#define __umulhi(a, b) ((uint32_t)(((uint64_t)(a) * (b)) >> 32))
#include "lbm_internal.hpp"

int main()
{
    int precision, n[3], outputs, face;
    uint64_t near, far;
    bool streamed;
    while (std::cin >> precision >> n[0] >> n[1] >> n[2] >> outputs >> face >> near >> far >>
           streamed) {
        lbm_solver s{};
        s.p.precision = precision;
        s.p.store_densities = s.p.store_velocities = outputs;
        s.n = 1;
        for (int i = 0; i < 3; i++) {
            s.size_h[i] = n[i] + 2;
            s.n *= n[i] + 2;
        }
        for (int i = 0; i < 6; i++)
            s.p.bc[i] = i == 2 ? face : (int)LBM_OBSTACLE;
        s.elem_bytes = precision == LBM_F32 ? 4 : precision == LBM_F64 ? 8 : 2;
        s.out_bytes = precision == LBM_F64 ? 8 : 4;
        std::cout << lbm::step_options(&s, 0, near << 20, far << 20, streamed) << ' '
                  << lbm::step_options(&s, 1, near << 20, far << 20, streamed) << '\n';
    }
    return 0;
}
