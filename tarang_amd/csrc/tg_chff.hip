// tg_chff.hip -- the Chebyshev (ChFF) path: Chebyshev along x, Fourier along
// y and z.  Line kernels over the (ky, kz) columns of the spectral layout
// (lx, ly, lz), lz fastest: one thread per column (or per column and parity for
// the Helmholtz solves), so that neighbouring threads read neighbouring lz and
// every step of the sequential recurrences along x is a coalesced access.  All
// arithmetic FP64.
#include "tg_device.h"
#include "tg_kernels.h"
#include "tg_chff.h"

namespace tg {

namespace {

__device__ __forceinline__ int kw(int l, int n) { return l <= n / 2 ? l : l - n; }

constexpr double kChEps = 1e-15;  // myconstant.MYEPS (Global.cc:62)

// Chebyshev derivative along x of E-double elements (E = 2 complex, 1 real):
// c_k b_k = b_{k+2} + 2 (k+1) a_{k+1}, k = N-2 .. 0, times kf.  The rows of
// eight steps are loaded together (one load at a time, its latency was the
// time: 19 us for a real 64 x 128 x 128 array, now 9).
template <int E>
__global__ void k_cheb_deriv(const double *__restrict__ A, double *__restrict__ B, int nx, size_t ncol, double kf)
{
    const size_t col = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= ncol) return;
    double b1[E], b2[E];
    for (int e = 0; e < E; e++) b1[e] = b2[e] = 0.0;
    for (int e = 0; e < E; e++) B[((size_t)(nx - 1) * ncol + col) * E + e] = 0.0;
    for (int k0 = nx - 2; k0 >= 0; k0 -= 8) {
        double a[8][E];
#pragma unroll
        for (int q = 0; q < 8; q++)
            for (int e = 0; e < E; e++) a[q][e] = A[((size_t)(max(k0 - q, 0) + 1) * ncol + col) * E + e];
        // (formed here: else each load would move to its step)
#pragma unroll
        for (int q = 0; q < 8; q++)
            for (int e = 0; e < E; e++) asm volatile("" : "+v"(a[q][e]));
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int k = k0 - q;
            if (k < 0) break;
            for (int e = 0; e < E; e++) {
                const double bk = b2[e] + (2.0 * (k + 1)) * a[q][e];
                b2[e] = b1[e];
                b1[e] = bk;
                B[((size_t)k * ncol + col) * E + e] = (k == 0 ? 0.5 * bk : bk) * kf;
            }
        }
    }
}

// Helmholtz_complex_full_array / Helmholtz_real_full_array (helmholtz.cc:
// 18-118): one parity of one column per thread, both parts of a complex
// element (E = 2; the matrix is the same), lambda = Kperp^2 + lam_sup, through
// Tridiagonal_solver (:155-231), Thual's algorithm: rows i = 1..m-1 of
// k = 2i + odd, first row all ones with value d0.  The right-hand side is R, or
// with VEL that of the momentum equation (BDF1.cc:80-110), ((N - V/dt) +
// grad_c p) / (-nu) of component c = comp + blockIdx.y, formed on the way down:
// the x-derivative of p is a sum from the top over the other parity, so it
// needs no pass of its own.
//
// Bound by the latency of the recurrence and of the rows' loads: a row takes
// one division (its coefficients' denominators, the same for all columns, are
// inverted once a block), eight rows are loaded together, the next eight while
// these are worked on, and X, Y lie in LDS (SCR: in memory, where a block's
// would pass 64 KB).  64 x 128 x 128: 40 us a solve, now 14, with the momentum equation's
// right-hand side (a pass of its own before) 20.
constexpr int kHelmThreads = 64, kHelmRows = 8;

template <int E, bool VEL, bool SCR>
__global__ void __launch_bounds__(kHelmThreads) k_helmholtz(HelmArgs a)
{
    extern __shared__ double sh[];
    const int N = a.g.nx, m = N / 2, n = m - 1;
    double *r1 = sh, *r2 = sh + N, *r3 = sh + 2 * N;
    for (int k = threadIdx.x; k < N; k += kHelmThreads) {
        r1[k] = k < 2 ? 0.0 : 1.0 / (4.0 * k * (k - 1));
        r2[k] = k < 2 ? 0.0 : 1.0 / (2.0 * ((double)k * k - 1));
        r3[k] = k < 2 ? 0.0 : 1.0 / (4.0 * k * (k + 1));
    }
    __syncthreads();
    const size_t ncol = (size_t)a.g.ny * a.g.nzc, nthr = 2 * ncol;
    const size_t t = (size_t)blockIdx.x * kHelmThreads + threadIdx.x;
    if (t >= nthr) return;
    const size_t col = t % ncol;
    const int odd = (int)(t / ncol);
    const int ly = (int)(col / a.g.nzc), lz = (int)(col % a.g.nzc);
    const double Ky = kw(ly, a.g.ny) * a.g.kf[1], Kz = lz * a.g.kf[2];
    const double kp2 = Ky * Ky + Kz * Kz;
    const int c = VEL ? a.comp + blockIdx.y : 0;
    double *__restrict__ U = VEL ? (c == 0 ? a.V[0] : c == 1 ? a.V[1] : a.V[2]) : a.U;
    const double *__restrict__ F = VEL ? (c == 0 ? a.N[0] : c == 1 ? a.N[1] : a.N[2]) : a.R;
    const double *__restrict__ P = a.P;
    auto row = [&](int i) { return ((size_t)(2 * i + odd) * ncol + col) * E; };
    double d0[E];
    for (int e = 0; e < E; e++) d0[e] = odd ? (a.vp[e] - a.vm[e]) / 2 : (a.vp[e] + a.vm[e]) / 2;
    if ((a.pressure_switch && kp2 < kChEps) || n <= 0) {
        // del^2 p = 0 at Kperp = 0: the linear profile through the wall values
        for (int i = 0; i < m; i++)
            for (int e = 0; e < E; e++) U[row(i) + e] = i == 0 ? d0[e] : 0.0;
        return;
    }
    // X(i), Y(i) of this thread
    double *Xs = SCR ? a.X + (size_t)blockIdx.y * nthr * m + t : sh + 3 * N + threadIdx.x;
    double *Ys = SCR ? a.Y + (size_t)blockIdx.y * nthr * m * E + t : sh + 3 * N + kHelmThreads * m + threadIdx.x;
    const size_t st = SCR ? nthr : kHelmThreads;
    const double lambda = kp2 + a.lam_sup, inv_dt = VEL ? 1 / a.dt : 0.0, inv_nu = VEL ? 1 / (-a.nu) : 0.0;
    const double Kc = c == 1 ? Ky : Kz;
    // the operands of kHelmRows rows from i down
    struct Rows {
        double f[kHelmRows][E], v[VEL ? kHelmRows : 1][E], p[VEL ? kHelmRows : 1][E];
    };
    auto load = [&](Rows &q, int i) {
#pragma unroll
        for (int s = 0; s < kHelmRows; s++) {
            const size_t r = row(max(i - s, 0));
            const int kp = 2 * max(i - s, 0) + odd + 1;   // x: the row above, of the other parity
            const size_t rp = c == 0 ? ((size_t)min(kp, N - 1) * ncol + col) * E : r;
#pragma unroll
            for (int e = 0; e < E; e++) {
                q.f[s][e] = F[r + e];
                if constexpr (VEL) {
                    q.v[s][e] = U[r + e];
                    q.p[s][e] = c == 0 && kp >= N ? 0.0 : P[rp + e];
                }
            }
        }
    };
    double up[E], mid[E], dx[E];   // F(i + 1), F(i); the derivative's sum
    double Xi = 0.0, Yi[E];
    for (int e = 0; e < E; e++) up[e] = mid[e] = dx[e] = Yi[e] = 0.0;
    auto step = [&](const Rows &q, int s, int i) {
        // low = F(i): solves row i + 1 from F(i), F(i + 1), F(i + 2)
        double low[E];
        if constexpr (VEL) {
            const int k = 2 * i + odd;
            double g[E];
            if (c == 0) {
                for (int e = 0; e < E; e++) {
                    dx[e] = dx[e] + (2.0 * (k + 1)) * q.p[s][e];
                    g[e] = (k == 0 ? 0.5 * dx[e] : dx[e]) * a.g.kf[0];
                }
            } else {
                g[0] = -Kc * q.p[s][E - 1];
                g[E - 1] = Kc * q.p[s][0];
            }
            for (int e = 0; e < E; e++) low[e] = ((q.f[s][e] - q.v[s][e] * inv_dt) + g[e]) * inv_nu;
        } else {
            for (int e = 0; e < E; e++) low[e] = q.f[s][e];
        }
        if (i < n) {
            const int k = 2 * (i + 1) + odd;
            const double ck = k == 2 ? 2.0 : 1.0, bk = k >= N - 2 ? 0.0 : 1.0, bk2 = k + 2 >= N - 2 ? 0.0 : 1.0;
            const double A = ck * lambda * r1[k], C = lambda * bk2 * r3[k];
            const double inv = 1.0 / (-(1 + lambda * bk * r2[k]) + C * Xi);
            for (int e = 0; e < E; e++) {
                const double d = ck * low[e] * r1[k] - bk * mid[e] * r2[k] + bk2 * up[e] * r3[k];
                Yi[e] = (d - C * Yi[e]) * inv;
                Ys[((size_t)i * E + e) * st] = Yi[e];
            }
            Xi = -A * inv;
            Xs[(size_t)i * st] = Xi;
        }
        for (int e = 0; e < E; e++) {
            up[e] = mid[e];
            mid[e] = low[e];
        }
    };
    Rows q0, q1;
    load(q0, n);
    for (int i0 = n; i0 >= 0; i0 -= 2 * kHelmRows) {
        if (i0 >= kHelmRows) load(q1, i0 - kHelmRows);
#pragma unroll
        for (int s = 0; s < kHelmRows; s++)
            if (i0 - s >= 0) step(q0, s, i0 - s);
        if (i0 >= 2 * kHelmRows) load(q0, i0 - 2 * kHelmRows);
#pragma unroll
        for (int s = 0; s < kHelmRows; s++)
            if (i0 - kHelmRows - s >= 0) step(q1, s, i0 - kHelmRows - s);
    }
    double theta = 1, THETA = 1, lam[E], LAM[E];
    for (int e = 0; e < E; e++) lam[e] = LAM[e] = 0.0;
#pragma unroll 8
    for (int i = 0; i < n; i++) {
        const double x = Xs[(size_t)i * st];
        theta = x * theta;
        THETA += theta;
        for (int e = 0; e < E; e++) {
            lam[e] = (x * lam[e]) + Ys[((size_t)i * E + e) * st];
            LAM[e] += lam[e];
        }
    }
    double y[E];
    for (int e = 0; e < E; e++) {
        y[e] = (d0[e] - LAM[e]) / THETA;
        U[row(0) + e] = y[e];
    }
#pragma unroll 8
    for (int i = 0; i < n; i++) {
        const double x = Xs[(size_t)i * st];
        for (int e = 0; e < E; e++) {
            y[e] = x * y[e] + Ys[((size_t)i * E + e) * st];
            U[row(i + 1) + e] = y[e];
        }
    }
}

// influence matrix (influence_matrix.cc:111-122)
__global__ void k_influence(const double *vxp, const double *vxm, double *M, int nx, size_t ncol, double kf)
{
    const size_t col = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= ncol) return;
    double m00 = 0, m01 = 0, m10 = 0, m11 = 0;
    for (int kx = 0; kx <= nx - 2; kx += 2) {
        const double f1 = (double)kx * kx, f2 = (double)(kx + 1) * (kx + 1);
        const size_t i0 = (size_t)kx * ncol + col, i1 = (size_t)(kx + 1) * ncol + col;
        m00 += f1 * vxp[i0] + f2 * vxp[i1];
        m01 += f1 * vxm[i0] + f2 * vxm[i1];
        m10 += (-f1) * vxp[i0] + f2 * vxp[i1];
        m11 += (-f1) * vxm[i0] + f2 * vxm[i1];
    }
    M[4 * col + 0] = m00 * kf;
    M[4 * col + 1] = m01 * kf;
    M[4 * col + 2] = m10 * kf;
    M[4 * col + 3] = m11 * kf;
}

// Compute_pressure_Ux_chebyshev (influence_matrix.cc:137-180).  The rows of 64
// columns are shared by the block's wavefronts (one thread a column left most
// of the chip idle: 51 us at 64 x 128 x 128, now 12).
constexpr int kInflWaves = 8;
__global__ void __launch_bounds__(64 * kInflWaves) k_influence_correct(InflArgs a)
{
    __shared__ cpx<double> sp[kInflWaves][64], sm[kInflWaves][64];
    const size_t ncol = (size_t)a.ny * a.nzc;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t at = (size_t)blockIdx.x * 64 + lane, col = at < ncol ? at : ncol - 1;
    cpx<double> dp = mk<double>(0, 0), dm = mk<double>(0, 0);
    cpx<double> *P = (cpx<double> *)a.P, *V1 = (cpx<double> *)a.V1;
#pragma unroll 4
    for (int kx = 2 * wave; kx <= a.nx - 2; kx += 2 * kInflWaves) {
        const double f1 = (double)kx * kx, f2 = (double)(kx + 1) * (kx + 1);
        const cpx<double> v0 = V1[(size_t)kx * ncol + col], v1 = V1[(size_t)(kx + 1) * ncol + col];
        dp = dp + (f1 * v0 + f2 * v1);
        dm = dm + ((-f1) * v0 + f2 * v1);
    }
    sp[wave][lane] = dp;
    sm[wave][lane] = dm;
    __syncthreads();
    dp = dm = mk<double>(0, 0);
    for (int w = 0; w < kInflWaves; w++) {
        dp = dp + sp[w][lane];
        dm = dm + sm[w][lane];
    }
    if (at >= ncol) return;
    const double vpt = a.M[4 * col], vmt = a.M[4 * col + 1], vpb = a.M[4 * col + 2], vmb = a.M[4 * col + 3];
    const double det = vpt * vmb - vmt * vpb;
    const cpx<double> vpp = a.kf * dp, vpm = a.kf * dm;
    cpx<double> delta_p = mk<double>(0, 0), delta_m = mk<double>(0, 0);
    if (fabs(det) > kChEps) {
        const cpx<double> np = vmt * vpm - vmb * vpp, nm = vpb * vpp - vpt * vpm;
        delta_p = mk<double>(np.x / det, np.y / det);
        delta_m = mk<double>(nm.x / det, nm.y / det);
    }
    const bool zero = col == 0;  // (ky, kz) = (0, 0): P and V1 set to zero
#pragma unroll 4
    for (int k = wave; k < a.nx; k += kInflWaves) {
        const size_t i = (size_t)k * ncol + col;
        const cpx<double> p = P[i] + (a.pp[i] * delta_p + a.pm[i] * delta_m);
        const cpx<double> v = V1[i] + (a.vxp[i] * delta_p + a.vxm[i] * delta_m);
        P[i] = mk<double>(zero ? 0.0 : p.x, zero ? 0.0 : p.y);
        V1[i] = mk<double>(zero ? 0.0 : v.x, zero ? 0.0 : v.y);
    }
}

__global__ void k_fill_double(double *a, size_t n, double v)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) a[i] = v;
}

__global__ void k_scale_real(double *a, size_t n, double s)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        a[i] = a[i] / s;
}

dim3 grid_for(size_t n, int threads = 256)
{
    size_t b = (n + threads - 1) / threads;
    if (b > 8192) b = 8192;
    return dim3((unsigned)(b ? b : 1));
}

}  // namespace

hipError_t launch_cheb_deriv(const Grid &g, const double *A, double *B, bool complex_, hipStream_t st)
{
    const size_t ncol = (size_t)g.ny * g.nzc;
    dim3 grid((unsigned)((ncol + 127) / 128));
    if (complex_) hipLaunchKernelGGL(k_cheb_deriv<2>, grid, dim3(128), 0, st, A, B, g.nx, ncol, g.kf[0]);
    else hipLaunchKernelGGL(k_cheb_deriv<1>, grid, dim3(128), 0, st, A, B, g.nx, ncol, g.kf[0]);
    return hipGetLastError();
}

hipError_t launch_helmholtz(const HelmArgs &a, hipStream_t st, int ncomp)
{
    const size_t nthr = (size_t)a.g.ny * a.g.nzc * 2, m = a.g.nx / 2;
    const dim3 grid((unsigned)((nthr + kHelmThreads - 1) / kHelmThreads), ncomp), block(kHelmThreads);
    const bool vel = a.P != nullptr;
    if ((a.E != 1 && a.E != 2) || (vel && a.E != 2) || (!vel && ncomp != 1)) return hipErrorInvalidValue;
    const size_t table = 3 * (size_t)a.g.nx * sizeof(double), lds = table + kHelmThreads * m * (1 + a.E) * sizeof(double);
    const bool scr = lds > 65536;
    const size_t shm = scr ? table : lds;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, shm, st, a); };
    if (a.E == 1) scr ? go(k_helmholtz<1, false, true>) : go(k_helmholtz<1, false, false>);
    else if (vel) scr ? go(k_helmholtz<2, true, true>) : go(k_helmholtz<2, true, false>);
    else scr ? go(k_helmholtz<2, false, true>) : go(k_helmholtz<2, false, false>);
    return hipGetLastError();
}

hipError_t launch_influence(const Grid &g, const double *vxp, const double *vxm, double *M, hipStream_t st)
{
    const size_t ncol = (size_t)g.ny * g.nzc;
    hipLaunchKernelGGL(k_influence, dim3((unsigned)((ncol + 127) / 128)), dim3(128), 0, st, vxp, vxm, M, g.nx, ncol,
                       g.kf[0]);
    return hipGetLastError();
}

hipError_t launch_influence_correct(const InflArgs &a, hipStream_t st)
{
    const size_t ncol = (size_t)a.ny * a.nzc;
    hipLaunchKernelGGL(k_influence_correct, dim3((unsigned)((ncol + 63) / 64)), dim3(64 * kInflWaves), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_fill_double(double *a, size_t n, double v, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_double, grid_for(n), dim3(256), 0, st, a, n, v);
    return hipGetLastError();
}

hipError_t launch_scale_real(double *a, size_t n, double divisor, hipStream_t st)
{
    hipLaunchKernelGGL(k_scale_real, grid_for(n), dim3(256), 0, st, a, n, divisor);
    return hipGetLastError();
}

}  // namespace tg
