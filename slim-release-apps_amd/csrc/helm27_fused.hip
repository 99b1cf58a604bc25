// The two operator applications of a complex64 BiCGStab iteration with every
// vector update fused in (epilogues 3 and 4 of the stencil body), for one
// vector: the work-list form of helm27_batch.hip without the list, with the
// updates and their scalars in FP64 and one rounding per stored vector, as the
// separate passes of bicgstab.hip have them (the batch rounds every product).
// An outer step of 25 iterations: 97 x 72 x 50 0.88 ms, 161 x 150 x 100 2.97,
// 240 x 240 x 140 6.9; with the updates in FP32 0.87, 2.95 and 6.8, with
// separate passes 1.44, 3.32 and 8.8.
#include "helm27_body.hpp"

namespace helm3d {

namespace {

// One shape, the one stencil_grid picks by rule: the block sums group the dots
// by the launch's blocks, so a shape tuned per handle would give two handles of
// one grid different inner solves.  Tiles of 64 x 4 in its place take, against
// 32 x 8, 100 to 102 % forward on nx x 72 x 50 for nx = 33 to 200 and 100 to 104 %
// adjoint, 97 % on 161 x 150 x 100, 98 % on 240 x 240 x 140 and 262 x 273 x 148, 110
// to 115 % on 220 x 180 x 120.
constexpr int kFTx = 32, kFTy = 8, kFPf = 2;

template <bool ADJ, bool WNC, int EPI>
__global__ __launch_bounds__(kFTx* kFTy) void helm27_fused_kernel(StencilLaunch<float> L)
{
    helm27_body<float, ADJ, false, WNC, kFTy, kFPf, EPI, 1, kFTx, double>(L, blockIdx.x, gridDim.x);
}

template <bool A, bool W, int EPI>
hipError_t launch_shape(const StencilLaunch<float>& L, const StencilGrid& g, hipStream_t s)
{
    hipLaunchKernelGGL((helm27_fused_kernel<A, W, EPI>), dim3(g.blocks), dim3(kFTx * kFTy), 0, s, L);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_stencil_fused(int variant, int epi, StencilLaunch<float> L, const StencilGrid& g, hipStream_t s)
{
    L.tiles_x = g.tiles_x;
    L.tiles_y = g.tiles_y;
    L.kchunk = g.kchunk;
    const bool adj = variant & VAR_ADJ, wnc = variant & VAR_WNC;
    if ((variant & VAR_DERIV) || (epi != 3 && epi != 4) || g.tx != kFTx || g.ty != kFTy || g.ry != 1)
        return hipErrorInvalidValue;
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
