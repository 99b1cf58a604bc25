// The two operator applications of a complex64 BiCGStab iteration with every
// vector update fused in (epilogues 3 and 4 of the stencil body), for one
// vector: the work-list form of helm27_batch.hip without the list.
#include "helm27_body.hpp"

namespace helm3d {

namespace {

template <bool ADJ, bool WNC, int TY, int PF, int EPI, int RY>
__global__ __launch_bounds__(TX* TY / RY) void helm27_fused_kernel(StencilLaunch<float> L)
{
    helm27_body<float, ADJ, false, WNC, TY, PF, EPI, RY>(L, blockIdx.x, gridDim.x);
}

template <bool A, bool W, int EPI>
hipError_t launch_shape(const StencilLaunch<float>& L, const StencilGrid& g, hipStream_t s)
{
    const dim3 grid(g.blocks);
    const bool two = g.pf >= 2;  // planes in flight: the four vectors of epilogue 3 leave registers for two
    if (g.ty == 8 && g.ry == 2) {
        if (two) hipLaunchKernelGGL((helm27_fused_kernel<A, W, 8, 2, EPI, 2>), grid, dim3(TX * 4), 0, s, L);
        else hipLaunchKernelGGL((helm27_fused_kernel<A, W, 8, 1, EPI, 2>), grid, dim3(TX * 4), 0, s, L);
    } else if (g.ty == 8) {
        if (two) hipLaunchKernelGGL((helm27_fused_kernel<A, W, 8, 2, EPI, 1>), grid, dim3(TX * 8), 0, s, L);
        else hipLaunchKernelGGL((helm27_fused_kernel<A, W, 8, 1, EPI, 1>), grid, dim3(TX * 8), 0, s, L);
    } else {
        if (two) hipLaunchKernelGGL((helm27_fused_kernel<A, W, 4, 2, EPI, 1>), grid, dim3(TX * 4), 0, s, L);
        else hipLaunchKernelGGL((helm27_fused_kernel<A, W, 4, 1, EPI, 1>), grid, dim3(TX * 4), 0, s, L);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_stencil_fused(int variant, int epi, StencilLaunch<float> L, const StencilGrid& g, hipStream_t s)
{
    L.tiles_x = g.tiles_x;
    L.tiles_y = g.tiles_y;
    L.kchunk = g.kchunk;
    const bool adj = variant & VAR_ADJ, wnc = variant & VAR_WNC;
    if ((variant & VAR_DERIV) || (epi != 3 && epi != 4)) return hipErrorInvalidValue;
    if (epi == 3) {
        if (!adj && !wnc) return launch_shape<false, false, 3>(L, g, s);
        if (!adj) return launch_shape<false, true, 3>(L, g, s);
        return wnc ? launch_shape<true, true, 3>(L, g, s) : launch_shape<true, false, 3>(L, g, s);
    }
    if (!adj && !wnc) return launch_shape<false, false, 4>(L, g, s);
    if (!adj) return launch_shape<false, true, 4>(L, g, s);
    return wnc ? launch_shape<true, true, 4>(L, g, s) : launch_shape<true, false, 4>(L, g, s);
}

}  // namespace helm3d
