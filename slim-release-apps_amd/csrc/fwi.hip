// FWI set-up and gradient support kernels.
//
//  * param2wavenum on the extended grid: the model on the physical grid is
//    extended into the PML by edge replication (opExtension.m:94-96 per axis,
//    composed in discrete_helmholtz.m:214-217 and applied at :240) and mapped
//    to wn = c v^-2 | c v | 1e-6 c v with c = (2 pi f)^2 and the derivatives
//    dwn, ddwn (param2wavenum.m:20-49).  One pass: each extended point reads
//    its clamped physical point (L2-resident along the PML slabs).
//  * the adjoint of the extension (opExtension.m:97-101 per axis): every
//    physical point sums the extended points that replicate it.  Interior
//    points have one preimage; face, edge and corner points sum their PML
//    line, sheet or block.
//  * a row-compressed operator with real weights for source injection and
//    receiver sampling (the sinc/Kaiser opInterp operators of DataGrid.m:22-44
//    reduce to a unit impulse on grid points, and are sparse in general).
//    Each output row is a gather, so the kernel needs no atomics; the host
//    builds the transposed rows for the injection direction.
#include <algorithm>
#include <type_traits>

#include "fwi.hpp"

namespace helm3d {

namespace {

constexpr int KB = 256;

__device__ inline int clampi(int a, int lo, int hi) { return a < lo ? lo : (a > hi ? hi : a); }

__global__ __launch_bounds__(KB) void param2wavenum_kernel(ExtGrid G, const double* __restrict__ v, int unit,
                                                           double c, double* __restrict__ wn,
                                                           double* __restrict__ dwn, double* __restrict__ ddwn)
{
    const long N = long(G.nt[0]) * G.nt[1] * G.nt[2];
    const long plane = long(G.nt[0]) * G.nt[1];
    for (long p = long(blockIdx.x) * KB + threadIdx.x; p < N; p += long(gridDim.x) * KB) {
        const int k = int(p / plane);
        const long r = p - long(k) * plane;
        const int j = int(r / G.nt[0]);
        const int i = int(r - long(j) * G.nt[0]);
        const int pi = clampi(i - G.lo[0], 0, G.np[0] - 1);
        const int pj = clampi(j - G.lo[1], 0, G.np[1] - 1);
        const int pk = clampi(k - G.lo[2], 0, G.np[2] - 1);
        const double m = v[pi + long(pj) * G.np[0] + long(pk) * G.np[0] * G.np[1]];
        double a, d, dd;
        if (unit == 0) {  // m/s
            const double iv = 1.0 / m;
            const double iv2 = iv * iv;
            a = c * iv2;
            d = -2.0 * c * iv2 * iv;
            dd = 6.0 * c * iv2 * iv2;
        } else {  // s2/m2 (c' = c) or s2/km2 (c' = 1e-6 c): linear in m
            a = c * m;
            d = c;
            dd = 0.0;
        }
        wn[p] = a;
        if (dwn) dwn[p] = d;
        if (ddwn) ddwn[p] = dd;
    }
}

// Preimage of physical index q along one axis: [q+lo] for interior points,
// [0, lo] for q = 0 and [q+lo, nt-1] for q = np-1 (both for np = 1).
__device__ inline void preimage(int q, int np, int lo, int nt, int& a, int& b)
{
    a = q == 0 ? 0 : q + lo;
    b = q == np - 1 ? nt - 1 : q + lo;
}

// Fold of the PML part.  Every extended point is read once, so the pass is
// bound by HBM; what has to be avoided is that the few physical points with a
// large preimage (a face point sums one PML line, an edge point a sheet, a
// corner a block: 21^3 points with a 20-point PML) are summed by one thread
// each.  Three kinds of blocks, the long ones first:
//   * face rows (j or k on a face of the physical box), one block per 64
//     interior x columns: the four waves take every fourth row of the
//     preimage, eight loads in flight, and are added in wave order;
//   * face rows, one block per x end point: the same, the lanes striding over
//     the end's segment of a row;
//   * interior rows, one wave per row: the interior columns are copied, the
//     two end points summed by the wave.
// 256 x 256 x 128 points + 20-point PML: 1372 us with one thread per physical
// point, 42 us so (184 MB moved).
constexpr int kFoldUnroll = 8;

__device__ inline double wave_sum_d(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__global__ __launch_bounds__(KB) void extension_adjoint_kernel(ExtGrid G, const double* __restrict__ gpml,
                                                               double* __restrict__ g, int accumulate, long nface,
                                                               int nchunk)
{
    __shared__ double red[KB];
    const int np0 = G.np[0], np1 = G.np[1], np2 = G.np[2];
    const long tplane = long(G.nt[0]) * G.nt[1];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const long b = blockIdx.x;
    const int nparts = nchunk + (np0 > 1 ? 2 : 1);
    if (b < nface * nparts) {
        // ---- a face row: all j of the k faces, then the j faces of the interior k
        const long f = b / nparts;
        const int part = int(b - f * nparts);
        const int kf = np2 > 1 ? 2 : 1, jf = np1 > 1 ? 2 : 1;
        int j, k;
        if (f < long(kf) * np1) {
            k = f < np1 ? 0 : np2 - 1;
            j = int(f < np1 ? f : f - np1);
        } else {
            const long q = f - long(kf) * np1;
            k = 1 + int(q / jf);
            j = (q % jf) ? np1 - 1 : 0;
        }
        int ja, jb, ka, kb;
        preimage(j, np1, G.lo[1], G.nt[1], ja, jb);
        preimage(k, np2, G.lo[2], G.nt[2], ka, kb);
        const int nj = jb - ja + 1;
        const long nrow = long(nj) * (kb - ka + 1);
        const double* base = gpml + long(ka) * tplane + long(ja) * G.nt[0];
        double* out = g + (long(k) * np1 + j) * np0;
        // row offsets of the preimage block, every fourth row: no division
        int jr = wid % nj;
        long kr = wid / nj;
        auto next_row = [&]() {
            const long o = kr * tplane + long(jr) * G.nt[0];
            jr += KB / 64;
            while (jr >= nj) {
                jr -= nj;
                ++kr;
            }
            return o;
        };
        const bool inner = part < nchunk;
        const int i = inner ? 1 + part * 64 + lane : (part == nchunk ? 0 : np0 - 1);
        int ia = i + G.lo[0], ib = ia;
        if (!inner) preimage(i, np0, G.lo[0], G.nt[0], ia, ib);
        const bool act = !inner || i < np0 - 1;
        double s = 0.0;
        // interior columns: one column per lane; end points: the lanes stride
        // over the end's segment of each row
        for (int ii = inner ? ia : ia + lane; act && ii <= ib; ii += 64) {
            const double* col = base + ii;
            jr = wid % nj;
            kr = wid / nj;
            long r = wid;
            for (; r + 4 * (kFoldUnroll - 1) < nrow; r += 4 * kFoldUnroll) {
                double v[kFoldUnroll];
#pragma unroll
                for (int u = 0; u < kFoldUnroll; ++u) v[u] = col[next_row()];
#pragma unroll
                for (int u = 0; u < kFoldUnroll; ++u) s += v[u];
            }
            for (; r < nrow; r += 4) s += col[next_row()];
        }
        if (!inner) s = wave_sum_d(s);
        red[threadIdx.x] = s;
        __syncthreads();
        if (wid == 0 && (inner ? act : lane == 0)) {
            const double t = (red[lane] + red[64 + lane]) + (red[128 + lane] + red[192 + lane]);
            out[i] = accumulate ? out[i] + t : t;
        }
        return;
    }
    // ---- interior rows: one wave each
    const long w = (b - nface * nparts) * (KB / 64) + wid;
    const int mj = np1 - 2, mk = np2 - 2;
    if (mj <= 0 || mk <= 0 || w >= long(mj) * mk) return;
    const int k = 1 + int(w / mj), j = 1 + int(w - long(k - 1) * mj);
    const double* row = gpml + long(k + G.lo[2]) * tplane + long(j + G.lo[1]) * G.nt[0];
    double* out = g + (long(k) * np1 + j) * np0;
    for (int i = 1 + lane; i < np0 - 1; i += 64) {
        const double t = row[i + G.lo[0]];
        out[i] = accumulate ? out[i] + t : t;
    }
#pragma unroll
    for (int end = 0; end < 2; ++end) {
        if (end == 1 && np0 == 1) break;
        const int i = end == 0 ? 0 : np0 - 1;
        int ia, ib;
        preimage(i, np0, G.lo[0], G.nt[0], ia, ib);
        double s = 0.0;
        for (int q = ia + lane; q <= ib; q += 64) s += row[q];
        s = wave_sum_d(s);
        if (lane == 0) out[i] = accumulate ? out[i] + s : s;
    }
}

// LPR lanes per stored row (a power of two up to a wave): the entries of a
// row are strided over its lanes and the lane sums added by a tree.
template <int LPR>
__global__ __launch_bounds__(KB) void csr_apply_kernel(int nrows, const long long* __restrict__ rowptr,
                                                       const long long* __restrict__ col,
                                                       const double* __restrict__ w,
                                                       const long long* __restrict__ oidx, double alpha,
                                                       const cpx<double>* __restrict__ in,
                                                       cpx<double>* __restrict__ out, int accumulate)
{
    const long t = long(blockIdx.x) * KB + threadIdx.x;
    const long r = t / LPR;
    if (r >= nrows) return;  // uniform over a row's lanes
    const int lane = int(t % LPR);
    double re = 0.0, im = 0.0;
    for (long long e = rowptr[r] + lane; e < rowptr[r + 1]; e += LPR) {
        const cpx<double> v = in[col[e]];
        re += w[e] * v.re;
        im += w[e] * v.im;
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) {
        re += __shfl_xor(re, o, LPR);
        im += __shfl_xor(im, o, LPR);
    }
    if (lane != 0) return;
    const long long o = oidx ? oidx[r] : r;
    cpx<double> y{alpha * re, alpha * im};
    if (accumulate) {
        y.re += out[o].re;
        y.im += out[o].im;
    }
    out[o] = y;
}

int grid_blocks(long n) { return int(std::min<long>(std::max<long>((n + KB - 1) / KB, 1), 8192)); }

}  // namespace

hipError_t launch_param2wavenum(const ExtGrid& G, const double* v, int unit, double c, double* wn, double* dwn,
                                double* ddwn, hipStream_t s)
{
    const long N = long(G.nt[0]) * G.nt[1] * G.nt[2];
    hipLaunchKernelGGL(param2wavenum_kernel, dim3(grid_blocks(N)), dim3(KB), 0, s, G, v, unit, c, wn, dwn, ddwn);
    return hipGetLastError();
}

hipError_t launch_extension_adjoint(const ExtGrid& G, const double* gpml, double* g, bool accumulate,
                                    hipStream_t s)
{
    const int nchunk = std::max(0, (G.np[0] - 2 + 63) / 64);
    const int nparts = nchunk + (G.np[0] > 1 ? 2 : 1);
    const long kf = G.np[2] > 1 ? 2 : 1, jf = G.np[1] > 1 ? 2 : 1;
    const long mj = std::max(0, G.np[1] - 2), mk = std::max(0, G.np[2] - 2);
    const long nface = kf * G.np[1] + jf * mk;
    const long blocks = nface * nparts + (mj * mk + KB / 64 - 1) / (KB / 64);
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(extension_adjoint_kernel, dim3(unsigned(blocks)), dim3(KB), 0, s, G, gpml, g,
                       int(accumulate), nface, nchunk);
    return hipGetLastError();
}

// Lanes per row by the row count alone (the entry counts are on the device):
// with few rows (receiver sampling, 512 entries a row off the grid) the chip
// is idle and a wave per row hides the chain of a long row; with many
// (injection onto the grid, mostly one entry a row) a lane per row is enough.
// 400 rows of 512 entries: 413 us with a lane per row, 12 us with a wave.
hipError_t launch_csr_apply(int nrows, const long long* rowptr, const long long* col, const double* w,
                            const long long* oidx, double alpha, const cpx<double>* in, cpx<double>* out,
                            bool accumulate, hipStream_t s)
{
    if (nrows <= 0) return hipSuccess;
    auto go = [&](auto lpr) {
        constexpr int L = decltype(lpr)::value;
        const long blocks = (long(nrows) * L + KB - 1) / KB;
        hipLaunchKernelGGL((csr_apply_kernel<L>), dim3(unsigned(blocks)), dim3(KB), 0, s, nrows, rowptr, col, w, oidx,
                           alpha, in, out, int(accumulate));
        return hipGetLastError();
    };
    if (nrows <= 16384) return go(std::integral_constant<int, 64>{});
    if (nrows <= 65536) return go(std::integral_constant<int, 8>{});
    return go(std::integral_constant<int, 1>{});
}

}  // namespace helm3d
