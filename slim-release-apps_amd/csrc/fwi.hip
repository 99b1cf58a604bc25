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

__device__ inline void csr_store(cpx<double>* out, long long o, double alpha, double re, double im, int accumulate)
{
    cpx<double> y{alpha * re, alpha * im};
    if (accumulate) {
        const cpx<double> p = out[o];
        y.re += p.re;
        y.im += p.im;
    }
    out[o] = y;
}

// One wave per stored row: the entries are strided over its lanes and the lane
// sums added by a tree.
__global__ __launch_bounds__(KB) void csr_row_kernel(int nrows, const long long* __restrict__ rowptr,
                                                     const long long* __restrict__ col,
                                                     const double* __restrict__ w,
                                                     const long long* __restrict__ oidx, double alpha,
                                                     const cpx<double>* __restrict__ in,
                                                     cpx<double>* __restrict__ out, int accumulate)
{
    const long r = long(blockIdx.x) * (KB / 64) + (threadIdx.x >> 6);
    if (r >= nrows) return;
    const int lane = threadIdx.x & 63;
    double re = 0.0, im = 0.0;
    for (long long e = rowptr[r] + lane; e < rowptr[r + 1]; e += 64) {
        const cpx<double> v = in[col[e]];
        re += w[e] * v.re;
        im += w[e] * v.im;
    }
    re = wave_sum_d(re);
    im = wave_sum_d(im);
    if (lane == 0) csr_store(out, oidx ? oidx[r] : r, alpha, re, im, accumulate);
}

// `per` (at most 64) consecutive stored rows per wave, lane l holding the ends
// of row l and, in the end, its sum.  How the wave works follows from its
// longest row: a lane per row up to 4 entries, 8 lanes per row up to 64, else
// the whole wave, row after row.
template <int L>
__device__ inline void csr_rows_by(int nr, int lane, long long e0, long long e1, const long long* __restrict__ col,
                                   const double* __restrict__ w, const cpx<double>* __restrict__ in, double& re,
                                   double& im)
{
    constexpr int G = 64 / L;  // rows at a time; those behind row nr - 1 are empty
    for (int q = 0; q < nr; q += G) {
        const int row = min(q + lane / L, 63);
        const long long b = __shfl(e0, row, 64), e = __shfl(e1, row, 64);
        double sr = 0.0, si = 0.0;
        for (long long t = b + lane % L; t < e; t += L) {
            const cpx<double> v = in[col[t]];
            sr += w[t] * v.re;
            si += w[t] * v.im;
        }
#pragma unroll
        for (int o = L / 2; o > 0; o >>= 1) {
            sr += __shfl_xor(sr, o, 64);
            si += __shfl_xor(si, o, 64);
        }
        const int k = lane - q;  // lane q + k takes the sum of the k-th group
        const double gr = __shfl(sr, (k * L) & 63, 64), gi = __shfl(si, (k * L) & 63, 64);
        if (k >= 0 && k < G) {
            re = gr;
            im = gi;
        }
    }
}

__global__ __launch_bounds__(KB) void csr_rows_kernel(int nrows, int per, const long long* __restrict__ rowptr,
                                                      const long long* __restrict__ col,
                                                      const double* __restrict__ w,
                                                      const long long* __restrict__ oidx, double alpha,
                                                      const cpx<double>* __restrict__ in,
                                                      cpx<double>* __restrict__ out, int accumulate)
{
    const int lane = threadIdx.x & 63;
    const long r0 = (long(blockIdx.x) * (KB / 64) + (threadIdx.x >> 6)) * per;
    if (r0 >= nrows) return;
    const int nr = int(min(long(per), nrows - r0));
    long long e0 = 0, e1 = 0;
    if (lane < nr) {
        e0 = rowptr[r0 + lane];
        e1 = rowptr[r0 + lane + 1];
    }
    const long long len = e1 - e0;
    double re = 0.0, im = 0.0;
    if (__any(len > 64)) csr_rows_by<64>(nr, lane, e0, e1, col, w, in, re, im);
    else if (__any(len > 4)) csr_rows_by<8>(nr, lane, e0, e1, col, w, in, re, im);
    else
        for (long long e = e0; e < e1; ++e) {
            const cpx<double> v = in[col[e]];
            re += w[e] * v.re;
            im += w[e] * v.im;
        }
    if (lane < nr) csr_store(out, oidx ? oidx[r0 + lane] : r0 + lane, alpha, re, im, accumulate);
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

// The host knows the row count, not the entry counts (they are on the device).
// Up to 4096 rows the chip is idle enough for a wave per row (receiver sampling,
// 512 entries a row off the grid: 400 rows 4.5 us, 4096 rows 16.3; a lane per row
// 325 and 333), one entry a row costing 2.4 us at 1000 rows and 3.2 at 4096 (a
// lane per row 2.4).  More rows go to about 3072 waves that look at their rows:
// 16384 rows of 1 / 64 / 512 entries 2.4 / 11.3 / 60.7 us, a lane per row 2.3 /
// 44.5 / 398, a wave per row 6.4 / 10.7 / 55.6.
hipError_t launch_csr_apply(int nrows, const long long* rowptr, const long long* col, const double* w,
                            const long long* oidx, double alpha, const cpx<double>* in, cpx<double>* out,
                            bool accumulate, hipStream_t s)
{
    if (nrows <= 0) return hipSuccess;
    constexpr int kWaves = KB / 64;
    if (nrows <= 4096) {
        hipLaunchKernelGGL(csr_row_kernel, dim3((nrows + kWaves - 1) / kWaves), dim3(KB), 0, s, nrows, rowptr, col, w,
                           oidx, alpha, in, out, int(accumulate));
        return hipGetLastError();
    }
    const int per = std::min(64, (nrows - 1) / 3072 + 1);
    const int waves = (nrows - 1) / per + 1;
    hipLaunchKernelGGL(csr_rows_kernel, dim3((waves - 1) / kWaves + 1), dim3(KB), 0, s, nrows, per, rowptr, col, w,
                       oidx, alpha, in, out, int(accumulate));
    return hipGetLastError();
}

}  // namespace helm3d
