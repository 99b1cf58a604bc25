// Work-list launches of the 27-point stencil: one launch applies the stencil
// to many (operator, vector) items, possibly on grids of different sizes
// (batched right-hand sides, several frequencies or models at once).
#include "helm27_body.hpp"

namespace helm3d {

namespace {

// One launch over a work list of stencil applications (possibly on different
// grids): item it owns blocks [first[it], first[it+1]); items with
// active[it] == 0 are skipped.  MIX: items marked narrow take tiles of half the
// columns and twice the rows (the same threads), the others TX x TY ones; a
// wave of a narrow tile is two rows, so only the y multipliers leave the scalar
// registers.  The choice is per item and per block, and the wide items of a
// mixed launch take as long as in a launch of their own.  The product at a point
// is the same for every shape; the partial sums of EPI 3 and 4 follow the
// item's blocks.
template <typename R, bool ADJ, bool DERIV, bool WNC, int TY, int PF, int EPI, int RY, bool MIX, int TXW>
__global__ __launch_bounds__(TXW* TY / RY) void helm27_batch_kernel(const StencilLaunch<R>* __restrict__ items,
                                                              const int* __restrict__ first, int nitems,
                                                              const int* __restrict__ active)
{
    const int bid = blockIdx.x;
    int lo = 0, hi = nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= bid) lo = mid;
        else hi = mid - 1;
    }
    if (active && !active[lo]) return;
    if constexpr (MIX) {
        if (items[lo].narrow) {
            helm27_body<R, ADJ, DERIV, WNC, 2 * TY, PF, EPI, RY, TXW / 2>(items[lo], bid - first[lo],
                                                                         first[lo + 1] - first[lo]);
            return;
        }
    }
    helm27_body<R, ADJ, DERIV, WNC, TY, PF, EPI, RY, TXW>(items[lo], bid - first[lo], first[lo + 1] - first[lo]);
}


template <typename R, bool A, bool W, int EPI>
hipError_t launch_b(const StencilLaunch<R>* items, const int* first, int nitems, int blocks, const int* active,
                    int ty, int pf, int ry, bool mix, hipStream_t s)
{
    const dim3 grid(blocks);
    if (mix) {
        hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 4, 2, EPI, 1, true, 64>), grid, dim3(TX * 4), 0, s, items,
                           first, nitems, active);
        return hipGetLastError();
    }
    if (ty == 8 && ry == 2) {
        if (pf >= 2)
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 8, 2, EPI, 2, false, 64>), grid, dim3(TX * 4), 0, s, items,
                               first, nitems, active);
        else
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 8, 1, EPI, 2, false, 64>), grid, dim3(TX * 4), 0, s, items,
                               first, nitems, active);
    } else if (ty == 8) {
        if (pf >= 2)
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 8, 2, EPI, 1, false, 32>), grid, dim3(32 * 8), 0, s, items,
                               first, nitems, active);
        else
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 8, 1, EPI, 1, false, 32>), grid, dim3(32 * 8), 0, s, items,
                               first, nitems, active);
    } else {
        if (pf >= 2)
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 4, 2, EPI, 1, false, 64>), grid, dim3(TX * 4), 0, s, items,
                               first, nitems, active);
        else
            hipLaunchKernelGGL((helm27_batch_kernel<R, A, false, W, 4, 1, EPI, 1, false, 64>), grid, dim3(TX * 4), 0, s, items,
                               first, nitems, active);
    }
    return hipGetLastError();
}

template <typename R, bool A, bool W>
hipError_t launch_v(int epi, const StencilLaunch<R>* items, const int* first, int nitems, int blocks,
                    const int* active, int ty, int pf, int ry, bool mix, hipStream_t s)
{
    switch (epi) {
    case 0: return launch_b<R, A, W, 0>(items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    case 1: return launch_b<R, A, W, 1>(items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    case 3: return launch_b<R, A, W, 3>(items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    case 4: return launch_b<R, A, W, 4>(items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

template <typename R>
hipError_t launch_stencil_batch(int variant, int epi, const StencilLaunch<R>* items, const int* first, int nitems,
                                int blocks, const int* active, int ty, int pf, hipStream_t s, int ry, bool mix)
{
    if (nitems <= 0 || blocks <= 0) return hipSuccess;
    if (variant & VAR_DERIV) return hipErrorInvalidValue;
    const bool adj = variant & VAR_ADJ, wnc = variant & VAR_WNC;
    if (!adj && !wnc) return launch_v<R, false, false>(epi, items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    if (!adj && wnc) return launch_v<R, false, true>(epi, items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    if (adj && !wnc) return launch_v<R, true, false>(epi, items, first, nitems, blocks, active, ty, pf, ry, mix, s);
    return launch_v<R, true, true>(epi, items, first, nitems, blocks, active, ty, pf, ry, mix, s);
}

template hipError_t launch_stencil_batch<double>(int, int, const StencilLaunch<double>*, const int*, int, int,
                                                 const int*, int, int, hipStream_t, int, bool);
template hipError_t launch_stencil_batch<float>(int, int, const StencilLaunch<float>*, const int*, int, int,
                                                const int*, int, int, hipStream_t, int, bool);

}  // namespace helm3d
