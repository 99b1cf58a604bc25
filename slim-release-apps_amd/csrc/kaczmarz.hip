// Kaczmarz row projections of the 27-point operator on gfx950.
//
// Reference semantics: do_sweep of Helm3dkaczswp_mex.c:60-117 -- for every
// row p of A (A = H, or H^H for the adjoint sweep),
//   d = omega (b_p - a_p . x) / |a_p|^2,   x_q += d conj(a_pq)  for the 27 q,
// visiting the rows forward and then backward (xyzloop_updown,
// Helm3d_27pt.h:63-108).  The lexicographic order is sequential; here the
// rows are ordered by 27 colours c = (i mod 3) + 3 (j mod 3) + 9 (k mod 3):
// rows of one colour touch disjoint 3x3x3 blocks, so one launch projects all
// of them at once, and colours 0..26 followed by 26..0 form the symmetric
// double sweep (its linear part Q keeps I - Q Hermitian, as CGMN requires).
// The iterates differ from the lexicographic sweep; the fixed point (A x = b)
// and the CGMN solution do not.
//
// Row coefficients are formed on the fly from the per-axis PML tables and wn
// (Helm3d_27pt.h:680-714 forward, :718-822 adjoint).  Complex wn is honoured
// (the reference's complex-wavenumber sweep gateway is built with a macro the
// header does not test and falls back to real wn; not reproduced).
#include <type_traits>

#include "helm27.hpp"

namespace helm3d {

namespace {

constexpr int KB = 256;

__device__ inline cpx<double> tab(const cpx<double>* t, int slot) { return t[slot]; }

// Stiffness coefficient coupling a point with PML values (lo, hi per axis)
// to its neighbour at offset d (Helm3d_27pt.h:680-714, non-mass terms):
//   centre -(c_x xi_x + c_y xi_y + c_z xi_z); face a: c_a xi_a^s + sum_{b!=a} w_ab xi_b;
//   edge (a,b): -w_ab (xi_a^s + xi_b^s) + w3a2 xi_c; corner -w3a2 sum xi^s.
__device__ inline cpx<double> stiff(const OpDesc<double>& op, int dx, int dy, int dz, const cpx<double> lo[3],
                                    const cpx<double> hi[3])
{
    const int d[3] = {dx, dy, dz};
    cpx<double> full[3], side[3];
    int nnz = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        full[a] = lo[a] + hi[a];
        side[a] = d[a] < 0 ? lo[a] : hi[a];
        nnz += d[a] != 0;
    }
    const double w[3][3] = {{0.0, op.xy, op.xz}, {op.xy, 0.0, op.yz}, {op.xz, op.yz, 0.0}};
    cpx<double> K{0.0, 0.0};
    if (nnz == 0) {
        K = -(op.c[0] * full[0] + op.c[1] * full[1] + op.c[2] * full[2]);
    } else if (nnz == 1) {
        const int a = d[0] ? 0 : (d[1] ? 1 : 2);
        K = op.c[a] * side[a];
#pragma unroll
        for (int b = 0; b < 3; ++b)
            if (b != a) K = rfma(K, w[a][b], full[b]);
    } else if (nnz == 2) {
        const int c = !d[0] ? 0 : (!d[1] ? 1 : 2);
        const int a = c == 0 ? 1 : 0, b = c == 2 ? 1 : 2;
        K = (-w[a][b]) * (side[a] + side[b]);
        K = rfma(K, op.w3a2, full[c]);
    } else {
        K = (-op.w3a2) * (side[0] + side[1] + side[2]);
    }
    return K;
}

__device__ inline double mass_mu(const OpDesc<double>& op, int nnz)
{
    return nnz == 0 ? op.wn_coef : (nnz == 1 ? -op.wm2 : (nnz == 2 ? -op.wm3 : -op.wm4));
}

__device__ inline cpx<double> wn_at(const OpDesc<double>& op, long q)
{
    if (op.wnc) return op.wnc[q];
    return cpx<double>{op.wn ? op.wn[q] : op.wn_const, 0.0};
}

// One thread per row of colour (ci, cj, ck) on a 3-D grid of 64 x 4 blocks
// (row index x along the lanes, one y row per wave, one z plane per grid
// layer).  The 27 coefficients and neighbour values are formed once and
// kept in registers: the 27 loads of a row issue together, and the update
// writes back x_q + d conj(a_pq) from the values already read (rows of a
// colour have disjoint supports, so no other row touches them).
template <bool ADJ>
__global__ __launch_bounds__(KB) void kacz_color_kernel(OpDesc<double> op, double omega, cpx<double>* __restrict__ x,
                                                         const cpx<double>* __restrict__ b, int ci, int cj, int ck,
                                                         int mx, int my)
{
    const int ti = int(blockIdx.x) * 64 + int(threadIdx.x & 63);
    const int tj = __builtin_amdgcn_readfirstlane(int(blockIdx.y) * 4 + int(threadIdx.x >> 6));
    const int tk = blockIdx.z;
    if (tj >= my) return;
    const bool act = ti < mx;  // lanes past the last row compute a copy and write nothing
    const int i = ci + 3 * min(ti, mx - 1), j = cj + 3 * tj, k = ck + 3 * tk;
    const int nx = op.nx, ny = op.ny, nz = op.nz;
    const long sy = nx, sz = long(nx) * ny;
    const long ip = i + j * sy + k * sz;
    // PML values at coordinate + d (d = -1, 0, 1) per axis; the forward row
    // uses only its own (d = 0), the adjoint row its neighbours'
    cpx<double> lo[3][3], hi[3][3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (!ADJ && d != 1) continue;
        lo[0][d] = tab(op.xlo, i + d); hi[0][d] = tab(op.xhi, i + d);
        lo[1][d] = tab(op.ylo, j + d); hi[1][d] = tab(op.yhi, j + d);
        lo[2][d] = tab(op.zlo, k + d); hi[2][d] = tab(op.zhi, k + d);
    }
    const cpx<double> wp = wn_at(op, ip);
    cpx<double> cf[27], xv[27];
    long qn[27];
    bool in[27];
#pragma unroll
    for (int n = 0; n < 27; ++n) {
        const int dx = n % 3 - 1, dy = (n / 3) % 3 - 1, dz = n / 9 - 1;
        const int a = i + dx, bb = j + dy, c = k + dz;
        in[n] = a >= 0 && a < nx && bb >= 0 && bb < ny && c >= 0 && c < nz;
        qn[n] = in[n] ? a + bb * sy + c * sz : ip;
        const int nnz = (dx != 0) + (dy != 0) + (dz != 0);
        cpx<double> v;
        if constexpr (!ADJ) {
            const cpx<double> l3[3] = {lo[0][1], lo[1][1], lo[2][1]}, h3[3] = {hi[0][1], hi[1][1], hi[2][1]};
            v = cmul(cpx<double>{mass_mu(op, nnz), 0.0}, wn_at(op, qn[n])) + stiff(op, dx, dy, dz, l3, h3);
        } else {
            // column p of H at row q, conjugated: xi of q, wn of p
            const cpx<double> l3[3] = {lo[0][dx + 1], lo[1][dy + 1], lo[2][dz + 1]};
            const cpx<double> h3[3] = {hi[0][dx + 1], hi[1][dy + 1], hi[2][dz + 1]};
            v = conjc(mass_mu(op, nnz) * wp + stiff(op, -dx, -dy, -dz, l3, h3));
        }
        cf[n] = in[n] ? v : cpx<double>{0.0, 0.0};
        xv[n] = x[qn[n]];
    }
    // residual of the row and |a|^2 (neighbours in the order dz, dy, dx)
    double atr = 0.0, ati = 0.0, nrm = 0.0;
#pragma unroll
    for (int n = 0; n < 27; ++n) {
        atr += cf[n].re * xv[n].re - cf[n].im * xv[n].im;
        ati += cf[n].re * xv[n].im + cf[n].im * xv[n].re;
        nrm += cf[n].re * cf[n].re + cf[n].im * cf[n].im;
    }
    const cpx<double> bp = b ? b[ip] : cpx<double>{0.0, 0.0};
    const double dr = omega * (bp.re - atr) / nrm, di = omega * (bp.im - ati) / nrm;
    // x_q += d conj(a_q)
#pragma unroll
    for (int n = 0; n < 27; ++n) {
        if (act && in[n] && (cf[n].re != 0.0 || cf[n].im != 0.0)) {
            cpx<double> v = xv[n];
            v.re += dr * cf[n].re + di * cf[n].im;
            v.im += di * cf[n].re - dr * cf[n].im;
            x[qn[n]] = v;
        }
    }
}

// ---- line form: the colours of one (j mod 3, k mod 3) class in one launch ----
//
// Rows (., j, k) and (., j', k') of one class touch disjoint sets of nine
// x lines, so a block that holds the nine lines of its (j, k) in LDS can run
// the x colours ci = 0, 1, 2 (or back, or both at the turn of the sweep) one
// after the other and write the lines back once: a double sweep moves x 17
// times instead of 54, with the projections of the colour form in the same
// order.
//
// Four lanes share a row, lane c taking the neighbours n = c, c + 4, ... of
// the 27 (n = dx + 1 + 3 (dy + 1) + 9 (dz + 1)): a projection is a chain of
// loads, a sum over the row, a division and the update, and a quarter of the
// row per lane shortens that chain and its registers (one lane per row holds
// 27 coefficients and 27 values: one wave per SIMD).  A coefficient is
// K_n + a_n X + mu_n wn: K_n, the y and z part, is fixed for the block and
// a_n, mu_n for the operator, so they are formed once per block (line_coef);
// X is the x PML value of the row (forward) or of its neighbour (adjoint), and
// as n mod 3 = (c + t) mod 3 at step t, each lane keeps its three X in the
// order in which it meets them.
//
// A double sweep, forward / adjoint, by colours and by lines: 240 x 240 x 140
// 6.22 / 4.80 and 1.55 / 1.47 ms (0.34 GB a launch; without the projections 50
// us each, with them 86), 84^3 582 / 485 and 199 / 185 us, 48 x 48 x 40 486 /
// 407 and 134 / 122 us.  Eight lanes per row: 1.95 / 1.95 ms, 212 / 199 and
// 122 / 117 us (more instructions in all); two: spills.
//
// The coefficients are grouped otherwise than in the colour form and omega /
// |a|^2 is one factor.  Against a double sweep in quad precision on the same
// tables, emulated on the host, the relative error is 7.5e-16 forward and 7.8e-16
// adjoint, the colour form's 8.5e-16 and 1.0e-15 (five grids of 24 x 24 x 20 to 84
// x 40 x 30).
constexpr int kLineThreads = 512;      // largest block
constexpr size_t kLineLds = 159 * 1024;  // LDS of a block (one kilobyte short of all of it)

struct LineCoef {
    cpx<double> K;
    double a, mu;
};

// Entry n of the block's coefficient table: the part of stiff() that carries
// the y and z PML, the weight of X and the mass weight.  Forward: PML values
// at (j, k).  Adjoint: those of the neighbour (j + dy, k + dz), from which the
// row's point lies at -d.  Zero where the neighbour's line is off the grid
// (and for n = 27, the padding of the fourth lane).
template <bool ADJ>
__device__ inline LineCoef line_coef(const OpDesc<double>& op, int n, int j, int k)
{
    LineCoef L{{0.0, 0.0}, 0.0, 0.0};
    const int dx = n % 3 - 1, dy = (n / 3) % 3 - 1, dz = n / 9 - 1;
    if (n >= 27 || j + dy < 0 || j + dy >= op.ny || k + dz < 0 || k + dz >= op.nz) return L;
    const int jy = ADJ ? j + dy : j, kz = ADJ ? k + dz : k;
    const cpx<double> yl = op.ylo[jy + 1], yh = op.yhi[jy + 1], zl = op.zlo[kz + 1], zh = op.zhi[kz + 1];
    const cpx<double> yf = yl + yh, zf = zl + zh;
    const cpx<double> ys = (ADJ ? dy > 0 : dy < 0) ? yl : yh, zs = (ADJ ? dz > 0 : dz < 0) ? zl : zh;
    const int nnz = (dx != 0) + (dy != 0) + (dz != 0);
    L.mu = mass_mu(op, nnz);
    if (dx == 0 && dy == 0 && dz == 0) {
        L.a = -op.c[0];
        L.K = -(op.c[1] * yf + op.c[2] * zf);
    } else if (dy == 0 && dz == 0) {
        L.a = op.c[0];
        L.K = op.xy * yf + op.xz * zf;
    } else if (dx == 0 && dz == 0) {
        L.a = op.xy;
        L.K = op.c[1] * ys + op.yz * zf;
    } else if (dx == 0 && dy == 0) {
        L.a = op.xz;
        L.K = op.c[2] * zs + op.yz * yf;
    } else if (dz == 0) {
        L.a = -op.xy;
        L.K = (-op.xy) * ys + op.w3a2 * zf;
    } else if (dy == 0) {
        L.a = -op.xz;
        L.K = (-op.xz) * zs + op.w3a2 * yf;
    } else if (dx == 0) {
        L.a = op.w3a2;
        L.K = (-op.yz) * (ys + zs);
    } else {
        L.a = -op.w3a2;
        L.K = (-op.w3a2) * (ys + zs);
    }
    return L;
}

// Sum over the four lanes of a row (quad permutes; every lane gets the sum,
// in the same order).
template <int CTRL>
__device__ inline double quad_swap(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp(int(b), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(int(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ inline double quad_sum(double v)
{
    v += quad_swap<0xB1>(v);  // lanes 1, 0, 3, 2
    v += quad_swap<0x4E>(v);  // lanes 2, 3, 0, 1
    return v;
}

// a, b or c for q = 0, 1, 2
__device__ inline cpx<double> pick(int q, cpx<double> a, cpx<double> b, cpx<double> c)
{
    return {q == 0 ? a.re : (q == 1 ? b.re : c.re), q == 0 ? a.im : (q == 1 ? b.im : c.im)};
}

// LDS of a block: the coefficient table, nine lines of x and, forward, of wn,
// with a zero column at either end (pitch nx + 2).
template <bool ADJ, bool WNC>
size_t line_lds(int nx)
{
    return 28 * sizeof(LineCoef) + size_t(9) * (nx + 2) * (16 + (ADJ ? 0 : (WNC ? 16 : 8)));
}

// seq: the x colours to run, two bits each, nseq of them.
template <bool ADJ, bool WNC>
__global__ __launch_bounds__(kLineThreads) __attribute__((amdgpu_waves_per_eu(4))) void kacz_line_kernel(OpDesc<double> op, double omega,
                                                                 cpx<double>* __restrict__ x,
                                                                 const cpx<double>* __restrict__ b, int cj, int ck,
                                                                 int seq, int nseq)
{
    extern __shared__ __align__(16) char lds[];
    const int nx = op.nx, ny = op.ny, nz = op.nz, pitch = nx + 2;
    LineCoef* tab_ = reinterpret_cast<LineCoef*>(lds);
    cpx<double>* sx = reinterpret_cast<cpx<double>*>(lds + 28 * sizeof(LineCoef));
    using W = std::conditional_t<WNC, cpx<double>, double>;
    W* sw = reinterpret_cast<W*>(sx + 9 * pitch);
    const W* wsrc = reinterpret_cast<const W*>(WNC ? static_cast<const void*>(op.wnc) : static_cast<const void*>(op.wn));
    const int j = cj + 3 * int(blockIdx.x), k = ck + 3 * int(blockIdx.y);
    const int tid = threadIdx.x, NT = blockDim.x;
    const long plane = long(nx) * ny;
    const long row0 = j * long(nx) + k * plane;

    // ---- the block's coefficients and the first row's operands are requested
    // ahead of the lines, so that the block waits for memory once
    LineCoef mine{};
    if (tid < 28) mine = line_coef<ADJ>(op, tid, j, k);
    // rows per thread and colour (1 up to 384 points a line)
    const int rstep = 3 * (NT >> 2);
    const int nr = (nx + rstep - 1) / rstep;

    // global operands of a row, loaded one row ahead
    struct Row {
        cpx<double> X0, X2, b;
        cpx<double> xl, xh;  // adjoint: the row's own PML values
        W w;                 // adjoint: the row's own wn
        int i;
    };
    auto load = [&](int s, int r) {
        Row R{};
        R.i = ((seq >> (2 * s)) & 3) + 3 * (tid >> 2) + r * rstep;
        const int ic = min(R.i, nx - 1);
        if constexpr (!ADJ) {
            R.X0 = op.xlo[ic + 1];
            R.X2 = op.xhi[ic + 1];
        } else {
            R.X0 = op.xhi[ic];
            R.X2 = op.xlo[ic + 2];
            R.xl = op.xlo[ic + 1];
            R.xh = op.xhi[ic + 1];
            R.w = wsrc[row0 + ic];
        }
        R.b = b ? b[row0 + ic] : cpx<double>{0.0, 0.0};
        return R;
    };
    Row N = load(0, 0);

    // ---- the nine lines, all loads of a thread in flight together
    bool in[9];
    long off[9];
#pragma unroll
    for (int l = 0; l < 9; ++l) {
        const int jj = j + l % 3 - 1, kk = k + l / 3 - 1;
        in[l] = jj >= 0 && jj < ny && kk >= 0 && kk < nz;
        off[l] = in[l] ? jj * long(nx) + kk * plane : row0;
    }
    for (int i = tid; i < nx; i += NT) {
        cpx<double> v[9];
        W w[9];
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            v[l] = x[off[l] + i];
            if constexpr (!ADJ) w[l] = wsrc[off[l] + i];
        }
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            sx[l * pitch + 1 + i] = in[l] ? v[l] : cpx<double>{0.0, 0.0};
            if constexpr (!ADJ) sw[l * pitch + 1 + i] = in[l] ? w[l] : W{};
        }
    }
    if (tid < 18) {
        const int e = (tid >> 1) * pitch + (tid & 1) * (nx + 1);
        sx[e] = cpx<double>{0.0, 0.0};
        if constexpr (!ADJ) sw[e] = W{};
    }
    if (tid < 28) tab_[tid] = mine;
    __syncthreads();

    const int c = tid & 3;
    const LineCoef* T = tab_ + c;  // entry t of the lane: T[4 * t]
    int at[7];
#pragma unroll
    for (int t = 0; t < 7; ++t) {
        const int n = c + 4 * t;
        at[t] = n < 27 ? (n / 3) * pitch + n % 3 : 4 * pitch + 1;  // position of (i + dx) is at + i
    }
    // x PML values of dx = -1, 0, 1 start at c mod 3 in this lane
    const int rot = c == 3 ? 0 : c;
    for (int s = 0; s < nseq; ++s) {
        for (int r = 0; r < nr; ++r) {
            const Row R = N;
            const bool wrap = r + 1 == nr;
            N = load(wrap ? min(s + 1, nseq - 1) : s, wrap ? 0 : r + 1);
            const int i = R.i;
            if (i >= nx) continue;  // uniform over the row's lanes
            cpx<double> cf[7], xv[7];
            W wv[7];
#pragma unroll
            for (int t = 0; t < 7; ++t) {
                xv[t] = sx[at[t] + i];
                if constexpr (!ADJ) wv[t] = sw[at[t] + i];
            }
            const cpx<double> X0 = R.X0, X2 = R.X2, Xf = ADJ ? R.xl + R.xh : R.X0 + R.X2;
            const cpx<double> Xa = pick(rot, X0, Xf, X2), Xb = pick(rot, Xf, X2, X0), Xc = pick(rot, X2, X0, Xf);
#pragma unroll
            for (int t = 0; t < 7; ++t) {
                const LineCoef L = T[4 * t];
                cpx<double> v = rfma(L.K, L.a, t % 3 == 0 ? Xa : (t % 3 == 1 ? Xb : Xc));
                if constexpr (!ADJ) {
                    if constexpr (WNC) v = rfma(v, L.mu, wv[t]);
                    else v.re = fma(L.mu, wv[t], v.re);
                } else {
                    if constexpr (WNC) v = rfma(v, L.mu, R.w);
                    else v.re = fma(L.mu, R.w, v.re);
                    v = conjc(v);
                }
                cf[t] = v;
            }
            if (i == 0 || i == nx - 1) {  // neighbours off the grid along x
#pragma unroll
                for (int t = 0; t < 7; ++t) {
                    const int d3 = (rot + t) % 3;  // dx + 1
                    const bool out = (i == 0 && d3 == 0) || (i == nx - 1 && d3 == 2);
                    cf[t].re = out ? 0.0 : cf[t].re;
                    cf[t].im = out ? 0.0 : cf[t].im;
                }
            }
            double atr = 0.0, ati = 0.0, nrm = 0.0;
#pragma unroll
            for (int t = 0; t < 7; ++t) {
                atr = fma(cf[t].re, xv[t].re, atr);
                ati = fma(cf[t].re, xv[t].im, ati);
                nrm = fma(cf[t].re, cf[t].re, nrm);
                atr = fma(-cf[t].im, xv[t].im, atr);
                ati = fma(cf[t].im, xv[t].re, ati);
                nrm = fma(cf[t].im, cf[t].im, nrm);
            }
            const double scale = omega / quad_sum(nrm);
            const double dr = scale * (R.b.re - quad_sum(atr)), di = scale * (R.b.im - quad_sum(ati));
            // x_q += d conj(a_q); off the grid the coefficient is zero and the
            // (zero) halo entry is written back
#pragma unroll
            for (int t = 0; t < 7; ++t) {
                xv[t].re = fma(dr, cf[t].re, fma(di, cf[t].im, xv[t].re));
                xv[t].im = fma(di, cf[t].re, fma(-dr, cf[t].im, xv[t].im));
                if (t < 6 || c < 3) sx[at[t] + i] = xv[t];
            }
        }
        __syncthreads();
    }

    for (int i = tid; i < nx; i += NT) {
#pragma unroll
        for (int l = 0; l < 9; ++l)
            if (in[l]) x[off[l] + i] = sx[l * pitch + 1 + i];
    }
}

// One colour class of rows (ci, cj, ck), the form without LDS lines.
hipError_t launch_color(bool adj, const OpDesc<double>& op, double omega, cpx<double>* x, const cpx<double>* b,
                        int ci, int cj, int ck, hipStream_t s)
{
    const int mx = (op.nx - ci + 2) / 3, my = (op.ny - cj + 2) / 3, mz = (op.nz - ck + 2) / 3;
    if (mx <= 0 || my <= 0 || mz <= 0) return hipSuccess;
    const dim3 grid(unsigned((mx + 63) / 64), unsigned((my + 3) / 4), unsigned(mz));
    if (adj)
        hipLaunchKernelGGL(kacz_color_kernel<true>, grid, dim3(KB), 0, s, op, omega, x, b, ci, cj, ck, mx, my);
    else
        hipLaunchKernelGGL(kacz_color_kernel<false>, grid, dim3(KB), 0, s, op, omega, x, b, ci, cj, ck, mx, my);
    return hipGetLastError();
}

// A run of x colours of the class (cj, ck).
template <bool ADJ, bool WNC>
hipError_t launch_line(const OpDesc<double>& op, double omega, cpx<double>* x, const cpx<double>* b, int cj, int ck,
                       int seq, int nseq, hipStream_t s)
{
    const int my = (op.ny - cj + 2) / 3, mz = (op.nz - ck + 2) / 3;
    if (my <= 0 || mz <= 0) return hipSuccess;
    const int nt = std::min(kLineThreads, ((op.nx + 2) / 3 * 4 + 63) / 64 * 64);
    const size_t lds = line_lds<ADJ, WNC>(op.nx);
    hipLaunchKernelGGL((kacz_line_kernel<ADJ, WNC>), dim3(unsigned(my), unsigned(mz)), dim3(unsigned(nt)), lds, s, op, omega, x, b, cj, ck, seq, nseq);
    return hipGetLastError();
}

}  // namespace

// nsweeps double sweeps: colours 0 .. 26 and back.  The line form runs while
// its nine lines fit in LDS (nx up to 747 forward, 1122 adjoint, 560 forward
// with complex wn), also where a compute unit holds one block only (740 x 80 x
// 60 forward 0.90 ms, by colours 2.21); longer lines take a launch per colour.
hipError_t launch_kacz_sweep(bool adj, const OpDesc<double>& op, double omega, cpx<double>* x,
                             const cpx<double>* b, int nsweeps, hipStream_t s)
{
    const bool wnc = op.wnc != nullptr;
    const size_t lds = adj ? line_lds<true, false>(op.nx)
                           : (wnc ? line_lds<false, true>(op.nx) : line_lds<false, false>(op.nx));
    const bool lines = lds <= kLineLds && (wnc || op.wn) && (op.nz + 2) / 3 <= 65535;
    // consecutive colours of one class (cj, ck), at most six: one launch
    int cls = -1, seq = 0, nseq = 0;
    auto flush = [&]() {
        if (nseq == 0) return hipSuccess;
        const int cj = cls % 3, ck = cls / 3;
        hipError_t e;
        if (adj)
            e = wnc ? launch_line<true, true>(op, omega, x, b, cj, ck, seq, nseq, s)
                    : launch_line<true, false>(op, omega, x, b, cj, ck, seq, nseq, s);
        else
            e = wnc ? launch_line<false, true>(op, omega, x, b, cj, ck, seq, nseq, s)
                    : launch_line<false, false>(op, omega, x, b, cj, ck, seq, nseq, s);
        seq = nseq = 0;
        return e;
    };
    for (int pass = 0; pass < 2 * nsweeps; ++pass) {
        for (int cc = 0; cc < 27; ++cc) {
            const int c = (pass & 1) ? 26 - cc : cc;
            if (!lines) {
                const hipError_t e = launch_color(adj, op, omega, x, b, c % 3, (c / 3) % 3, c / 9, s);
                if (e != hipSuccess) return e;
                continue;
            }
            if (c / 3 != cls || nseq == 6) {
                const hipError_t e = flush();
                if (e != hipSuccess) return e;
                cls = c / 3;
            }
            seq |= (c % 3) << (2 * nseq++);
        }
    }
    return flush();
}

}  // namespace helm3d
