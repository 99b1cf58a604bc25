// Launch interface of the stencil and Krylov kernels (internal to the library).
#pragma once

#include <algorithm>

#include "helm3d_common.hpp"

namespace helm3d {

// Operator variant bits; the six combinations built as MEX binaries in
// ibin/install_MEX:88-105 are {0, ADJ} x {real wn, WNC, DERIV}.
enum Variant : int { VAR_FORW = 0, VAR_ADJ = 1, VAR_DERIV = 2, VAR_WNC = 4 };

template <typename R>
struct StencilLaunch {
    OpDesc<R> op;
    const cpx<R>* x;     // input vector (device, interleaved complex)
    cpx<R>* y;           // output: y = alpha * (H x) + beta * b
    const cpx<R>* b;     // optional addend (nullptr: none)
    R alpha, beta;
    const double* anrm;  // optional (EPI 0/1): alpha is divided by sqrt(*anrm) (device scalar)
    double* norm_part;   // optional: per-block partial sums of |y|^2
    // optional FWI-gradient epilogue: instead of storing y, accumulate
    // gg[phys] += gscale * Re(conj(gu) * y) over the physical box
    // [p0, p0+pn) of each axis (comp2phys truncation of the PML).
    const cpx<R>* gu;
    double* gg;
    double gscale;
    int p0[3], pn[3];
    // write-only sink of kSinkSlots values for steps/lanes with no output
    cpx<R>* sink;
    int tiles_x, tiles_y, kchunk;
    // fused BiCGStab forms, scalars in sc:
    //   EPI 3: f0 = r, f1 = p, f2 = v, f3 = t of the previous iteration;
    //          y = new v, o2 = new p, o3 = new r, zz = z (updated in place),
    //          rh = rhat
    //   EPI 4: f0 = r, f1 = v; y = t, rh = rhat
    const cpx<R>* f0;
    const cpx<R>* f1;
    const cpx<R>* f2;
    const cpx<R>* f3;
    cpx<R>* o2;
    cpx<R>* o3;
    cpx<R>* zz;
    const cpx<R>* rh;
    double* sc;
    int rho_new, rho_old, first;
    int narrow;       // mixed work lists: 32 x 8 tiles
    const int* skip;  // optional (device): the launch does nothing while *skip != 0
};

struct GmresDevState;

// Arnoldi step of GMRES on small grids (EPI 5): y = H x /
// ||x||, then the dots of y with the basis slots, in one launch.
//   npart, npn  partial sums of ||x||^2, added by every wave in one order
//               (npart = nullptr: y = H x, and the fields up to tol unused)
//   nrm, row    ||x||^2 stored by block 0 for the update pass and the least
//               squares (row optional)
//   start       0: an inner step; 1: first step of a solve, 2: of a restarted
//               cycle: block 0 opens the state st, and the launch does nothing
//               on a zero residual (1) or one below tol (2)
//   V, ldv, k   basis slots 0 .. k-1 (k <= kStepMaxK)
//   dpart       partials of the 2k sums: dpart[q * blocks + block]
constexpr int kStepMaxK = 8;
template <typename R>
struct StepArgs {
    const double* npart;
    int npn;
    int start;
    double* nrm;
    double* row;
    GmresDevState* st;
    double tol;
    const cpx<R>* V;
    long ldv;
    int k;
    double* dpart;
};

// Launch shape: tx x ty column tiles, z chunks of kchunk planes, pf planes of
// loads in flight, ry rows per thread (2 only with ty = 8).
constexpr int kSinkSlots = 65536;

struct StencilGrid {
    int tiles_x, tiles_y, kchunk, nchunks, blocks, ty, pf, ry, tx;
};

// z planes per block (even) for a launch over `tiles` columns of nz planes.  A
// block marches its planes and two halo planes, blocks run `slots` at a time,
// and the launch ends with a tail in which slots idle, longer when the last
// round is nearly empty:
//   cost(kc) = tiles (nz + halo chunks) / slots
//            + (kc + fill) (wait + tail (ceil(x) - x)),  x = blocks / slots,
// fitted to launches of chunks from 2 planes to the whole column on 36 grids of
// 31 x 31 x 19 to 420 x 400 x 150 with rotating inputs (complex128 48 x 48 x 40:
// 2 planes 6.0 us, 8 planes 9.7; 84^3: 6 planes 11.9, 9 planes 16.3, 42 planes
// 34.0).  In complex128 the same constants do not serve both ends: three blocks
// of 256 threads fit a compute unit, and grids of more than 100 tiles want longer
// chunks than a fit over all finds (best of the sweep 100 %: 187 x 203 x 111 20
// planes 108 %, 28 planes 105; 200 x 200 x 100 20 planes 113, 26 planes 100; 240
// x 240 x 140 24 planes 105, 48 planes 100; mean over 16 such grids 105.5 and
// 101.5).
struct ChunkCost {
    int slots;
    double halo, fill, wait, tail;
};
constexpr ChunkCost kCost64{512, 2, 2, 0.2, 0.15}, kCost64Large{768, 4, 0, 0.15, 0.15}, kCost64Resid{512, 1, 2, 0, 0.25},
    kCost32{1024, 2, 2, 0.2, 0.15};
constexpr int kLargeTiles = 100;
int stencil_chunk(long tiles, int nz, const ChunkCost& m);

// kchunk <= 0 picks the chunk by stencil_chunk for precision R; ty in {4, 8};
// pf in 1..4; ry in {1, 2} (2 needs ty = 8; otherwise 1 is used); tx = 0: tiles
// of 32 columns, of 64 with two rows per thread.  Tiles of 32 x 8 read 1.33
// points per output and waste no more than 31 lanes of a row, tiles of 64 x 4
// with the same threads 1.55 and 63; and more waves lie outside the PML.
// Against 64 x 4 in about 480 blocks, both with the chunk by their rule,
// complex128 / complex64 forward on rotating inputs: 84^3 14.4 -> 11.9 / 11.1 ->
// 9.9 us, 160 x 160 x 80 26.1 -> 21.8 / 20.0 -> 15.7, 240 x 240 x 140 82.5 -> 79.7 /
// 59.7 -> 50.7, 280 x 280 x 140 108 -> 95 / 69.9 -> 61.4; 250 x 100 x 60 19.7 ->
// 21.3 (100 tiles of 64 x 4 made 500 equal blocks).
template <typename R>
StencilGrid stencil_grid(int nx, int ny, int nz, int kchunk, int ty = 8, int pf = 2, int ry = 1, int tx = 0);

// The shape by rule of the wavenumber-derivative forms (gradient epilogue among
// them).  They hold no PML sums and wait for memory, so grids of more than 100
// column tiles take few long chunks, about 480 blocks in all: derivative matvec
// in complex128 forward / adjoint and gradient on 240 x 240 x 140 with the chunk
// of the operator 72.7 / 63.4 and 90.5 us, so 67.0 / 58.0 and 83.4; 296 x 296 x
// 168 in complex64 126.9 / 118.3, so 114.7 / 107.7.  Smaller grids keep the
// operator's chunk (120 x 110 x 90: 10.9 us with 10 planes, 11.4 with 12).
template <typename R>
StencilGrid stencil_deriv_grid(int nx, int ny, int nz);

// The shape by rule of the complex128 residual form (b - H x).  With the addend
// in flight two blocks fit a compute unit and an uneven last round costs more;
// its constants find the best chunk of the sweep on eight grids of 84^3 to 280 x
// 280 x 140.  They are used from the size at which the operator's differ (240 x
// 240 x 140: 48 planes 115.8 us, 70 planes 93.9; 187 x 203 x 111: 28 planes 61.5,
// 37 planes 50.9; 64 x 4 tiles in 480 blocks 98.2 and 57.2).
StencilGrid stencil_resid_grid(int nx, int ny, int nz);

template <typename R>
hipError_t launch_stencil(int variant, StencilLaunch<R> L, const StencilGrid& g, hipStream_t s);

// The Arnoldi step form (EPI 5, no DERIV).
template <typename R>
hipError_t launch_stencil_step(int variant, StencilLaunch<R> L, const StepArgs<R>& X, const StencilGrid& g,
                               hipStream_t s);

// The fused BiCGStab forms (epi 3 or 4, no DERIV) for one vector.
hipError_t launch_stencil_fused(int variant, int epi, StencilLaunch<float> L, const StencilGrid& g, hipStream_t s);

// One launch over nitems device-resident StencilLaunch items (operators
// without DERIV); item it owns blocks [first[it], first[it+1]) of `blocks`,
// launched with its own tiles_x/tiles_y/kchunk and the common shape (ty, pf,
// ry: two rows per thread with ty = 8).
// epi: 0 (y = alpha H x), 1 (+ beta b), 3, 4 (fused BiCGStab forms).
// mix: items with narrow set have tiles of 32 columns by 8 rows, the others 64
// by 4 (ty, pf, ry unused).  Otherwise all items have 64 x ty tiles, or 32 x 8
// for ty = 8 with one row per thread.
// active (nullable): items with active[it] == 0 do nothing.
template <typename R>
hipError_t launch_stencil_batch(int variant, int epi, const StencilLaunch<R>* items, const int* first, int nitems,
                                int blocks, const int* active, int ty, int pf, hipStream_t s, int ry = 1, bool mix = false);

}  // namespace helm3d
