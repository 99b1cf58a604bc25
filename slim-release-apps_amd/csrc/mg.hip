// Grid transfers of the multigrid V-cycle (construct_multigrid.m:30-40):
// prolongation = trilinear interpolation between the PML-extended grids of two
// levels, both spanning linspace(0,1,n) per axis (fine2coarse.m:40-57 with
// LinInterp1D.m), restriction = 1/8 times its transpose.  Per axis the host
// supplies, for every fine index, the coarse bracket I and the weights of I
// and I+1, and for every coarse index the list of fine indices that use it
// (row-compressed), so both directions are gathers.  Sums are formed in FP64
// for complex128 and complex64 vectors alike.
#include "mg.hpp"

namespace helm3d {

namespace {

constexpr int KB = 256;

// The transfers run on a 3-D grid of 64 x 4 thread blocks (x along the lanes,
// one y row per wave): no index division, and the y and z table entries are
// uniform over a wave.

// xf += P xc at fine points: the 2 x 2 x 2 coarse neighbours of the bracket.  A
// thread takes kProlongPlanes points along z, their loads issued together (120 x
// 120 x 70 to 240 x 240 x 140, complex64: one point 58.5 us, four 54.2).
constexpr int kProlongPlanes = 4;
template <typename R>
__global__ __launch_bounds__(KB) void prolong_add_kernel(MgAxes T, const cpx<R>* __restrict__ xc,
                                                         cpx<R>* __restrict__ xf)
{
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = __builtin_amdgcn_readfirstlane(int(blockIdx.y) * 4 + int(threadIdx.x >> 6));
    const int kz = blockIdx.z * kProlongPlanes;
    if (j >= T.nf[1]) return;
    const int ic = min(i, T.nf[0] - 1);
    const long ncx = T.nc[0], ncxy = long(T.nc[0]) * T.nc[1];
    const int Ix = T.ax[0].I[ic], Iy = T.ax[1].I[j];
    const double wx[2] = {T.ax[0].wa[ic], T.ax[0].wb[ic]};
    const double wy[2] = {T.ax[1].wa[j], T.ax[1].wb[j]};
    const int jx[2] = {Ix, min(Ix + 1, T.nc[0] - 1)};
    const long jy[2] = {Iy * ncx, min(Iy + 1, T.nc[1] - 1) * ncx};
    const long nfxy = long(T.nf[0]) * T.nf[1], pf = ic + long(j) * T.nf[0];
    cpx<R> v[kProlongPlanes][8], o[kProlongPlanes];
    double wz[kProlongPlanes][2];
#pragma unroll
    for (int u = 0; u < kProlongPlanes; ++u) {
        const int k = min(kz + u, T.nf[2] - 1);
        const int Iz = T.ax[2].I[k];
        wz[u][0] = T.ax[2].wa[k];
        wz[u][1] = T.ax[2].wb[k];
        const long jz[2] = {Iz * ncxy, min(Iz + 1, T.nc[2] - 1) * ncxy};
        o[u] = xf[pf + k * nfxy];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int a = 0; a < 2; ++a) v[u][4 * c + 2 * b + a] = xc[jx[a] + jy[b] + jz[c]];
    }
#pragma unroll
    for (int u = 0; u < kProlongPlanes; ++u) {
        double re = 0.0, im = 0.0;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const double wyz = wy[b] * wz[u][c];
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const double w = wx[a] * wyz;
                    re = fma(w, double(v[u][4 * c + 2 * b + a].re), re);
                    im = fma(w, double(v[u][4 * c + 2 * b + a].im), im);
                }
            }
        if (i < T.nf[0] && kz + u < T.nf[2])
            xf[pf + (kz + u) * nfxy] = cpx<R>{R(double(o[u].re) + re), R(double(o[u].im) + im)};
    }
}

// yc = scale * P^T rf at coarse points: per (z, y) entry of the transposed
// lists (uniform over the wave), the x entries of the lane's coarse index
// from the padded list (at most 8 entries, the padded width read at run time),
// so the loads of a coarse point are independent and issued together.
constexpr int kGatherWidth = 8;
template <typename R>
__global__ __launch_bounds__(KB) void restrict_kernel(MgAxes T, double scale, const cpx<R>* __restrict__ rf,
                                                      cpx<R>* __restrict__ yc)
{
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = __builtin_amdgcn_readfirstlane(int(blockIdx.y) * 4 + int(threadIdx.x >> 6));
    const int k = blockIdx.z;
    if (j >= T.nc[1]) return;
    const int ic = min(i, T.nc[0] - 1);
    const long nfx = T.nf[0], nfxy = long(T.nf[0]) * T.nf[1];
    const int pw = T.ax[0].pw;
    int fx[kGatherWidth];
    double wxv[kGatherWidth];
#pragma unroll
    for (int e = 0; e < kGatherWidth; ++e) {
        fx[e] = e < pw ? T.ax[0].pfi[long(ic) * pw + e] : 0;
        wxv[e] = e < pw ? T.ax[0].pfw[long(ic) * pw + e] : 0.0;
    }
    double re = 0.0, im = 0.0;
    const int z0 = T.ax[2].rp[k], z1 = T.ax[2].rp[k + 1];
    const int y0 = T.ax[1].rp[j], y1 = T.ax[1].rp[j + 1];
    for (int ez = z0; ez < z1; ++ez) {
        const long fz = T.ax[2].fi[ez] * nfxy;
        const double wz = T.ax[2].fw[ez];
        for (int ey = y0; ey < y1; ++ey) {
            const long base = T.ax[1].fi[ey] * nfx + fz;
            const double wyz = wz * T.ax[1].fw[ey];
            double sr = 0.0, si = 0.0;
#pragma unroll
            for (int e = 0; e < kGatherWidth; ++e) {
                if (e < pw) {
                    const cpx<R> v = rf[base + fx[e]];
                    sr = fma(wxv[e], double(v.re), sr);
                    si = fma(wxv[e], double(v.im), si);
                }
            }
            re = fma(wyz, sr, re);
            im = fma(wyz, si, im);
        }
    }
    if (i < T.nc[0]) yc[i + long(j) * T.nc[0] + long(k) * T.nc[0] * T.nc[1]] = cpx<R>{R(scale * re), R(scale * im)};
}

// The same sums with the y and z weights applied first: a wave's run of coarse
// points of a row uses at most 128 consecutive fine columns, so it adds the
// weighted fine rows of the window column by column -- coalesced loads, two
// columns a lane, each fine value read once per row instead of once per x
// entry -- and takes the x entries from LDS at the end.  The gather above moves
// WX x 64 strided values through L1 per fine row (240 x 240 x 140 to 120 x 120
// x 70, complex64: 56.3 us; here 43.5, every fine row read by two or three
// coarse rows and planes through L2).  Window positions behind the last fine
// column repeat it and are not used.
template <typename R, int WY>
__global__ __launch_bounds__(KB) void restrict_window_kernel(MgAxes T, double scale, const cpx<R>* __restrict__ rf,
                                                             cpx<R>* __restrict__ yc)
{
    __shared__ double sre[KB / 64][kRestrictWindow], sim[KB / 64][kRestrictWindow];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int run = T.ax[0].run;
    const int i0 = blockIdx.x * run, i = i0 + lane;
    const int j = min(int(blockIdx.y) * 4 + wv, T.nc[1] - 1);
    const int k = blockIdx.z;
    const long nfx = T.nf[0], nfxy = long(T.nf[0]) * T.nf[1];
    const MgAxis &ax = T.ax[0], &ay = T.ax[1], &az = T.ax[2];
    const int f0 = ax.fi[ax.rp[i0]];  // lists ascend: the window's first column
    const long c0 = min(long(f0 + lane), nfx - 1), c1 = min(long(f0 + 64 + lane), nfx - 1);
    const int y0 = ay.rp[j], ny = ay.rp[j + 1] - y0;
    long fy[WY];
    double wy[WY];
#pragma unroll
    for (int e = 0; e < WY; ++e) {
        fy[e] = e < ny ? ay.fi[y0 + e] * nfx : 0;
        wy[e] = e < ny ? ay.fw[y0 + e] : 0.0;
    }
    double r0 = 0.0, m0 = 0.0, r1 = 0.0, m1 = 0.0;
    const int z0 = az.rp[k], z1 = az.rp[k + 1];
    for (int ez = z0; ez < z1; ++ez) {
        const cpx<R>* __restrict__ pz = rf + az.fi[ez] * nfxy;
        const double wz = az.fw[ez];
        cpx<R> a[WY], b[WY];
#pragma unroll
        for (int e = 0; e < WY; ++e) {
            if (e < ny) {
                a[e] = pz[fy[e] + c0];
                b[e] = pz[fy[e] + c1];
            }
        }
#pragma unroll
        for (int e = 0; e < WY; ++e) {
            if (e < ny) {
                const double w = wz * wy[e];
                r0 = fma(w, double(a[e].re), r0);
                m0 = fma(w, double(a[e].im), m0);
                r1 = fma(w, double(b[e].re), r1);
                m1 = fma(w, double(b[e].im), m1);
            }
        }
    }
    sre[wv][lane] = r0;
    sim[wv][lane] = m0;
    sre[wv][lane + 64] = r1;
    sim[wv][lane + 64] = m1;
    __syncthreads();
    if (lane >= run || i >= T.nc[0] || int(blockIdx.y) * 4 + wv >= T.nc[1]) return;
    double re = 0.0, im = 0.0;
    for (int q = ax.rp[i]; q < ax.rp[i + 1]; ++q) {
        const int p = ax.fi[q] - f0;
        re = fma(ax.fw[q], sre[wv][p], re);
        im = fma(ax.fw[q], sim[wv][p], im);
    }
    yc[i + long(j) * T.nc[0] + long(k) * T.nc[0] * T.nc[1]] = cpx<R>{R(scale * re), R(scale * im)};
}

dim3 transfer_grid(const int n[3]) { return dim3((n[0] + 63) / 64, (n[1] + 3) / 4, n[2]); }

}  // namespace

template <typename R>
hipError_t launch_prolong_add(const MgAxes& T, const cpx<R>* xc, cpx<R>* xf, hipStream_t s)
{
    dim3 g = transfer_grid(T.nf);
    g.z = (g.z + kProlongPlanes - 1) / kProlongPlanes;
    hipLaunchKernelGGL(prolong_add_kernel<R>, g, dim3(KB), 0, s, T, xc, xf);
    return hipGetLastError();
}

template <typename R>
hipError_t launch_restrict(const MgAxes& T, double scale, const cpx<R>* rf, cpx<R>* yc, hipStream_t s)
{
    // a ratio of 2 always fits the window; the gather takes ratios from about 3.9
    // along x (a run of 32 coarse points no longer fits) and those along y whose
    // lists exceed the window's 8 rows; beyond 8 entries along x (ratio 4 and
    // more) neither does
    if (T.ax[0].run > 0 && T.ax[0].pw <= 8 && T.ax[1].pw <= 8) {
        const dim3 gw((T.nc[0] + T.ax[0].run - 1) / T.ax[0].run, (T.nc[1] + 3) / 4, T.nc[2]);
        if (T.ax[1].pw <= 4)
            hipLaunchKernelGGL((restrict_window_kernel<R, 4>), gw, dim3(KB), 0, s, T, scale, rf, yc);
        else if (T.ax[1].pw == 5)
            hipLaunchKernelGGL((restrict_window_kernel<R, 5>), gw, dim3(KB), 0, s, T, scale, rf, yc);
        else
            hipLaunchKernelGGL((restrict_window_kernel<R, 8>), gw, dim3(KB), 0, s, T, scale, rf, yc);
        return hipGetLastError();
    }
    if (T.ax[0].pw < 1 || T.ax[0].pw > kGatherWidth) return hipErrorInvalidValue;
    hipLaunchKernelGGL(restrict_kernel<R>, transfer_grid(T.nc), dim3(KB), 0, s, T, scale, rf, yc);
    return hipGetLastError();
}

template hipError_t launch_prolong_add<double>(const MgAxes&, const cpx<double>*, cpx<double>*, hipStream_t);
template hipError_t launch_prolong_add<float>(const MgAxes&, const cpx<float>*, cpx<float>*, hipStream_t);
template hipError_t launch_restrict<double>(const MgAxes&, double, const cpx<double>*, cpx<double>*, hipStream_t);
template hipError_t launch_restrict<float>(const MgAxes&, double, const cpx<float>*, cpx<float>*, hipStream_t);

}  // namespace helm3d
