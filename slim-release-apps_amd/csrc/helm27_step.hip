// Arnoldi steps of the device-driven GMRES on small grids: matvec and dots in
// one launch (EPI 5 of the stencil body).  On a coarse multigrid level a launch
// takes a few microseconds whatever it does, so the step is two launches (this
// and the update pass) instead of four: the norm of the input is summed from
// the update pass's partials here, the dots from this launch's partials there.
// What is left is one chain of dependent loads and exchanges: the partials and
// the skip flag are read behind the first plane loads, and the dots read two
// planes of outputs and basis together (FWI objective: 180 -> 174 ms).
#include "helm27_body.hpp"

namespace helm3d {

namespace {

// One shape, the one stencil_grid picks by rule: the dots are grouped by the
// launch's blocks, and their bits must follow the grid alone.
constexpr int kSTx = 32, kSTy = 8, kSPf = 2;

template <typename R, bool ADJ, bool WNC>
__global__ __launch_bounds__(kSTx* kSTy) void helm27_step_kernel(StencilLaunch<R> L, StepArgs<R> X)
{
    helm27_body<R, ADJ, false, WNC, kSTy, kSPf, 5, 1, kSTx>(L, blockIdx.x, gridDim.x, &X);
}

template <typename R, bool A, bool W>
hipError_t launch_shape(const StencilLaunch<R>& L, const StepArgs<R>& X, const StencilGrid& g, hipStream_t s)
{
    hipLaunchKernelGGL((helm27_step_kernel<R, A, W>), dim3(g.blocks), dim3(kSTx * kSTy), 0, s, L, X);
    return hipGetLastError();
}

}  // namespace

template <typename R>
hipError_t launch_stencil_step(int variant, StencilLaunch<R> L, const StepArgs<R>& X, const StencilGrid& g,
                               hipStream_t s)
{
    L.tiles_x = g.tiles_x;
    L.tiles_y = g.tiles_y;
    L.kchunk = g.kchunk;
    if ((variant & VAR_DERIV) || X.k < 1 || X.k > kStepMaxK || g.tx != kSTx || g.ty != kSTy || g.ry != 1)
        return hipErrorInvalidValue;
    const bool adj = variant & VAR_ADJ, wnc = variant & VAR_WNC;
    if (!adj && !wnc) return launch_shape<R, false, false>(L, X, g, s);
    if (!adj) return launch_shape<R, false, true>(L, X, g, s);
    return wnc ? launch_shape<R, true, true>(L, X, g, s) : launch_shape<R, true, false>(L, X, g, s);
}

template hipError_t launch_stencil_step<double>(int, StencilLaunch<double>, const StepArgs<double>&,
                                                const StencilGrid&, hipStream_t);
template hipError_t launch_stencil_step<float>(int, StencilLaunch<float>, const StepArgs<float>&,
                                               const StencilGrid&, hipStream_t);

}  // namespace helm3d
