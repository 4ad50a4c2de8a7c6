// lxw2d.hip -- Lax-Wendroff time-integrated fluxes (ConstructIntegratedR,
// lib/2d/ConstructIntegratedR.cpp:59-296) on the extended grid
// [-3, mx+2] x [-3, my+2] that the following WENO stage reads.
#include <hip/hip_runtime.h>
#include "kernels.h"
#include "lxw_body.h"

namespace finess {

template <class P, typename R, int TI, int TJ>
__global__ __launch_bounds__(TI* TJ) void k_lxw_flux(LxwArgs a, int ntj)
{
    __shared__ LxwSmem<TI, TJ, P::MEQN, R> sm;
    if (lxw_halted(a)) return;
    const int ti = blockIdx.x / ntj, tj = blockIdx.x - ti * ntj;
    const int e0i = ti * TI, e0j = tj * TJ;
    lxw_phase_load<P, TI, TJ, R>(threadIdx.x, TI * TJ, e0i, e0j, a, sm);
    __syncthreads();
    lxw_phase_cell<P, TI, TJ, R>(threadIdx.x, e0i, e0j, a, sm);
}

// The FP64 form other than the limited step's.  It moves 505 MB at 2048^2 (the
// state in, F and G out) in 135 us where the hyper-dual form took 264: bound
// by FP64 issue and the latency of its loads together (164 registers and 42 KB
// of LDS, three workgroups per CU; asking for two or four waves per SIMD made
// no difference).
template <class P, int TI, int TJ>
__global__ __launch_bounds__(TI* TJ) __attribute__((amdgpu_waves_per_eu(3))) void k_lxw_flux64(LxwArgs a, int ntj)
{
    __shared__ LxwSmem64<P, TI, TJ> sm;
    if (lxw_halted(a)) return;
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int ti = tile / ntj, tj = tile - ti * ntj;
    const int e0i = ti * TI, e0j = tj * TJ;
    const bool nz = lxw64_load<P, TI, TJ>(threadIdx.x, e0i, e0j, a, sm);
    // a tile without rho w takes the form that leaves its derivatives out
    if (P::MEQN == 5 && !__syncthreads_or(nz)) {
        lxw64_cell<P, TI, TJ, true>(threadIdx.x, e0i, e0j, a, sm);
        return;
    }
    if (P::MEQN != 5) __syncthreads();
    lxw64_cell<P, TI, TJ, false>(threadIdx.x, e0i, e0j, a, sm);
}

template <class P>
static int launch_flux64(const LxwArgs& a, hipStream_t st)
{
    constexpr int TI = 8, TJ = 32;
    const int nti = (a.mx + 6 + TI - 1) / TI, ntj = (a.my + 6 + TJ - 1) / TJ;
    hipLaunchKernelGGL((k_lxw_flux64<P, TI, TJ>), dim3(nti * ntj), dim3(TI * TJ), 0, st, a, ntj);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// fp32: the FP32 stencil form (Euler), whose Lax-Wendroff stage reads the
// fluxes as FP32: differences, hyper-dual products and Taylor terms in FP32.
int launch_lxw_flux(int physics, int fp32, const LxwArgs& a, hipStream_t st)
{
    if (!fp32 && physics == PHYS_EULER && !a.limited) return launch_flux64<Euler2D>(a, st);
    if (!fp32 && physics == PHYS_SHALLOW_WATER) return launch_flux64<ShallowWater2D>(a, st);
    constexpr int TI = 8, TJ = 32;
    const int nti = (a.mx + 6 + TI - 1) / TI, ntj = (a.my + 6 + TJ - 1) / TJ;
    if (physics == PHYS_EULER && fp32)
        hipLaunchKernelGGL((k_lxw_flux<Euler2D, float, TI, TJ>), dim3(nti * ntj), dim3(TI * TJ), 0, st, a, ntj);
    else if (physics == PHYS_EULER)
        hipLaunchKernelGGL((k_lxw_flux<Euler2D, double, TI, TJ>), dim3(nti * ntj), dim3(TI * TJ), 0, st, a, ntj);
    else
        return -1;
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

} // namespace finess
