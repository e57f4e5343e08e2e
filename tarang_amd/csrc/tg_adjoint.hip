// tg_adjoint.hip -- adjoint of the NS right-hand side f(V) = -P NL(D V),
// NL_i = sum_j i K_j F[u_j u_i], u = I(D V), and of the Lawson RK4 step.
// (No counterpart in the reference.)
//
// Inner product: the real dot product of the stored half-spectrum (Re, Im).
// With c = 1 on the kz = 0 and kz = Nz/2 planes and 2 elsewhere the
// transposes of the transforms are I^T = N^3 diag(c) F and
// F^T = N^-3 I diag(1/c); (i K)^T = -i K; P and D are symmetric.  So
//   f'(V)^T G = -D diag(c) F[q],  q_m = sum_j u_j sigma_jm,
//   sigma_jm = I(diag(1/c)(-i K_m M_j - i K_j M_m)),  M = P G,
// which needs the stage's u (taped by the forward sweep), five inverse and
// three forward transforms: x-inverse of the symmetrised fields (built from
// M in registers), y-inverse, z c2r + products with the tape + r2c,
// y-forward, x-forward with the stage epilogue.  sigma is trace-free
// (sigma_jj summed is -2i K.M/c = 0, M being projected), so sigma_zz =
// -sigma_xx - sigma_yy is not transformed: the z pass subtracts u_z sigma_xx
// and u_z sigma_yy from q_z instead.
#include "tg_adjoint.h"
#include "tg_device.h"
#include "tg_pass.h"

namespace tg {

struct XsymArgs {
    const double *G[3];
    void *S[5];
    const void *tw;
    Grid g;
};

// From a column's cotangent m (consumed): M = P G, the five symmetrised fields
// xx, yy, xy, yz, zx of (-i K_m M_j - i K_j M_m)/c (zz = -xx - yy), their
// x-inverse, stored into S.  Pad columns carry zeros.
template <bool NT, typename T, int L, int CB>
__device__ __forceinline__ void xsym_columns(const Grid &g, const ColTile<T, L, CB> &t, const ColX<T, L, CB> &x,
                                             const cpx<T> *tw, void *const *S, cpx<double> (*m)[8])
{
    constexpr int TPL = L / 8;
    constexpr bool NTW = NT && CB * sizeof(cpx<T>) >= 128;
    const double Ky = kwave(t.ly, g.ny) * g.kf[1], Kz = t.lz * g.kf[2];
    {
        // M = P G (Pressure.cc:56-72 form: G - K (K.G)/K^2, identity at K = 0)
        const int jh = hidden(t.j);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const double Kx = kwave(jh + TPL * s, g.nx) * g.kf[0];
            const double ks = (Kx * Kx + Ky * Ky) + Kz * Kz;
            if (ks > 0.0) {
                cpx<double> d = Kx * m[0][s];
                d = d + Ky * m[1][s];
                d = d + Kz * m[2][s];
                const cpx<double> e = mk<double>(d.x / ks, d.y / ks);
                m[0][s] = m[0][s] - Kx * e;
                m[1][s] = m[1][s] - Ky * e;
                m[2][s] = m[2][s] - Kz * e;
            }
            settle(m[0][s]);
            settle(m[1][s]);
            settle(m[2][s]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    const double w = !t.live ? 0.0 : (t.lz == 0 || t.lz == g.nz / 2) ? 1.0 : 0.5;
    constexpr int pa[5] = {0, 1, 0, 1, 2};
    constexpr int pb[5] = {0, 1, 1, 2, 0};
#pragma unroll
    for (int p = 0; p < 5; p++) {
        cpx<T> v[8];
        const int jh = hidden(t.j);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const double Kx = kwave(jh + TPL * s, g.nx) * g.kf[0];
            const double K[3] = {Kx, Ky, Kz};
            const cpx<double> A = m[pa[p]][s], B = m[pb[p]][s];
            // -i K_b A - i K_a B, times 1/c
            const double re = K[pb[p]] * A.y + K[pa[p]] * B.y;
            const double im = -(K[pb[p]] * A.x + K[pa[p]] * B.x);
            v[s] = mk<T>((T)(w * re), (T)(w * im));
        }
        fft_exchange<L, +1>(v, x, tw, jh);
        pin_memory_order();
        if (t.inside) col_store<NTW>(v, (cpx<T> *)S[p] + t.cw0, t.stepw, t.offt);
    }
}

// Column tiles in registers in transform order (ColX), as k_xfwd_adj.
template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8), 2) k_xinv_sym(XsymArgs a)
{
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, false)) return;
    const ColTile<T, L, CB> t(g, tile);
    cpx<double> m[3][8];
#pragma unroll
    for (int c = 0; c < 3; c++) col_load<false>(m[c], (const cpx<double> *)a.G[c] + t.state0, t.steps, t.offs);
    for (int i = threadIdx.x; i < L; i += CB * (L / 8)) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    xsym_columns<false>(g, t, X{lds + t.c}, tw, a.S, m);
}

// q += u * v (SUB: q -= u * v) on the packed real points of this thread (u
// from the tape line).
template <typename T, int M, bool SUB = false>
__device__ __forceinline__ void tape_mac(cpx<T> *q, const cpx<T> *v, const cpx<T> *__restrict__ u, int j)
{
    constexpr int TPL = M / 8;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const cpx<T> A = u[j + TPL * s];
        const cpx<T> d = mk<T>(A.x * v[s].x, A.y * v[s].y);
        q[s] = SUB ? q[s] - d : q[s] + d;
    }
}

// sigma lines in a.in[]: 0 xx, 1 yy, 2 xy, 3 yz, 4 zx (zz = -xx - yy).  The
// three accumulators q_m = sum_j u_j sigma_jm are live together, so each
// sigma line takes one c2r: a diagonal line sigma_jj adds u_j sigma_jj to q_j
// and, as its share of sigma_zz, subtracts u_z sigma_jj from q_z; an
// off-diagonal line sigma_jm adds u_j sigma_jm to q_m and u_m sigma_jm to
// q_j.  Five c2r and three r2c per line.
template <typename T, int M, bool NT, int W>
__global__ void __launch_bounds__(64 * W) k_z_adj(ZArgs a)
{
    constexpr int TPL = M / 8;
    constexpr int LPB = ZLines<M, W>::LPB;
    constexpr int LP = lpad_len(M);
    __shared__ cpx<T> lds[LPB * LP], ldw[2 * M];
    const ZTwiddles<T, M> tw(ldw, a.twm, a.twn);
    const ZLines<M, W> z(a.g);
    if (z.spare) return;
    // (formed anew for powers of two: from z's members the compiler no longer
    // moved the tape's loads ahead of the transforms, 485 us a launch at 256^3
    // FP64 against 357)
    constexpr bool WHOLE = 64 % TPL == 0;
    const int li = WHOLE ? threadIdx.x / TPL : z.li, j = WHOLE ? threadIdx.x % TPL : z.j;
    const size_t line = (size_t)blockIdx.x * LPB + li, nlines = (size_t)a.g.nx * a.g.ny;
    const bool valid = line < nlines;
    const size_t lsafe = valid ? line : nlines - 1;
    cpx<T> *L = lds + li * LP;
    const size_t off = lsafe * a.g.nzp;
    cpx<T> q[3][8];
#pragma unroll
    for (int m = 0; m < 3; m++)
#pragma unroll
        for (int s = 0; s < 8; s++) q[m][s] = mk<T>(0, 0);
#pragma unroll 1
    for (int t = 0; t < 5; t++) {
        // sigma_jm of line t: (j, m) = (t, t) for t < 2, (t-2, t-1 mod 3) after
        const int jt = t < 2 ? t : t - 2, mt = t < 2 ? t : (t == 4 ? 0 : t - 1);
        const cpx<T> *X = (const cpx<T> *)(t == 0 ? a.in[0] : t == 1 ? a.in[1] : t == 2 ? a.in[2] :
                                            t == 3 ? a.in[3] : a.in[4]);
        cpx<T> v[8];
        zline_c2r<T, M, NT>(v, X + off, L, tw, j);
        line_sync();
        const cpx<T> *uj = (const cpx<T> *)(jt == 0 ? a.tape[0] : jt == 1 ? a.tape[1] : a.tape[2]) + lsafe * M;
        const cpx<T> *um = (const cpx<T> *)(mt == 0 ? a.tape[0] : mt == 1 ? a.tape[1] : a.tape[2]) + lsafe * M;
        const cpx<T> *uz = (const cpx<T> *)a.tape[2] + lsafe * M;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (k == mt) tape_mac<T, M>(q[k], v, uj, j);
            if (t >= 2 && k == jt) tape_mac<T, M>(q[k], v, um, j);
        }
        if (t < 2) tape_mac<T, M, true>(q[2], v, uz, j);
    }
#pragma unroll
    for (int m = 0; m < 3; m++) {
        cpx<T> *Q = (cpx<T> *)(m == 0 ? a.out[0] : m == 1 ? a.out[1] : a.out[2]);
        zline_r2c_post<T, M, NT>(q[m], Q + off, L, tw, j, valid, a.g.nzp - M);
    }
}

struct XadjArgs {
    void *Q[3];
    double *lam[3], *acc[3], *lg[3];
    void *S[5];  // FUSE: the next stage's five symmetrised fields
    const void *tw;
    Grid g;
    AdjParams ap;
};

// FUSE: the next stage's cotangent (lg, or lam after the step's last stage)
// stays in registers instead of going through HBM, and the next stage's
// xsym_columns runs on it here (lg is not stored).
// Bound by HBM: columns go from memory to registers and back in transform
// order, one instance per mode (its loads and factors only); with the tiles
// staged through LDS a launch at 256^3 FP64 took 732 us, now 590 (S1; 4.0 TB/s).
template <typename T, int L, int CB, int MODE, bool FUSE, bool NT>
__global__ void __launch_bounds__(CB *(L / 8), 2) k_xfwd_adj(XadjArgs a)
{
    constexpr int TPL = L / 8, NTH = CB * TPL;
    constexpr bool NTW = NT && CB * sizeof(cpx<T>) >= 128;
    constexpr bool NEED_L = MODE != ADJ_RHS, NEED_A = MODE == ADJ_S2 || MODE == ADJ_S1 || MODE == ADJ_S0;
    constexpr bool EH = MODE == ADJ_S3 || MODE == ADJ_S2 || MODE == ADJ_S1, E1 = MODE == ADJ_S1 || MODE == ADJ_S0;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    // exp(-nu K^2 dt/2) and exp(-nu K^2 dt) at this thread's points
    __shared__ double visc[(EH ? 1 : 0) + (E1 ? 1 : 0) + (EH || E1 ? 0 : 1)][8 * NTH];
    const Grid &g = a.g;
    const AdjParams &ap = a.ap;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, false)) return;
    const ColTile<T, L, CB> t(g, tile);
    const int j = t.j;
    cpx<T> v[8];
    cpx<double> lm[8], ac[8];
    col_load<NTW>(v, (const cpx<T> *)a.Q[0] + t.cw0, t.stepw, t.offt);
    if (NEED_L) col_load<false>(lm, (const cpx<double> *)a.lam[0] + t.state0, t.steps, t.offs);
    if (NEED_A) col_load<false>(ac, (const cpx<double> *)a.acc[0] + t.state0, t.steps, t.offs);
    for (int i = threadIdx.x; i < L; i += NTH) tw[i] = ((const cpx<T> *)a.tw)[i];
    if (EH || E1) {
        const double Ky = kwave(t.ly, g.ny) * g.kf[1], Kz = t.lz * g.kf[2];
#pragma unroll 2
        for (int s = 0; s < 8; s++) {
            const double Kx = kwave(j + TPL * s, g.nx) * g.kf[0];
            const double ks = (Kx * Kx + Ky * Ky) + Kz * Kz;
            const double kp = hyper_power(ap.hq, ks);
            if (EH) visc[0][s * NTH + threadIdx.x] = exp((ap.fh + ap.fhh * kp) * ks);
            if (E1) visc[EH ? 1 : 0][s * NTH + threadIdx.x] = exp((ap.f1 + ap.f1h * kp) * ks);
        }
    }
    lds_barrier();
    const X x{lds + t.c};
    int zx0, zx1;
    dealias_rows(g, t.ly, t.lz, zx0, zx1);
    const double cw = (t.lz == 0 || t.lz == g.nz / 2) ? -1.0 : -2.0;
    const double c_sixth = (1.0 / 6) * ap.dt, c_third = (1.0 / 3) * ap.dt, c_half = 0.5 * ap.dt;
    cpx<double> gn[3][8];   // the next cotangent
#pragma unroll
    for (int K = 0; K < 3; K++) {
        const int jh = hidden(j);
        fft_exchange<L, -1>(v, x, tw, jh);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            cpx<double> r = ap.scale * cvt<double>(v[s]);
            r = lx >= zx0 && lx <= zx1 ? mk<double>(0, 0) : cw * r;
            const double Eh = EH ? visc[0][s * NTH + threadIdx.x] : 0.0;
            const double Ef = E1 ? visc[EH ? 1 : 0][s * NTH + threadIdx.x] : 0.0;
            cpx<double> nx;
            if constexpr (MODE == ADJ_RHS) {
                nx = r;
            } else if constexpr (MODE == ADJ_S3) {
                const cpx<double> lv = c_sixth * r;
                ac[s] = (Eh * Eh) * lv;
                nx = c_third * (Eh * lm[s]) + ap.dt * (Eh * lv);
            } else if constexpr (MODE == ADJ_S2) {
                ac[s] = ac[s] + Eh * r;
                nx = c_third * (Eh * lm[s]) + c_half * r;
            } else if constexpr (MODE == ADJ_S1) {
                ac[s] = ac[s] + Eh * r;
                nx = c_sixth * (Ef * lm[s]) + c_half * (Eh * r);
            } else {
                nx = (Ef * lm[s] + ac[s]) + r;
            }
            gn[K][s] = nx;
            settle(gn[K][s]);
            __builtin_amdgcn_sched_barrier(0);
        }
        pin_memory_order();
        if (K < 2) col_load<NTW>(v, (const cpx<T> *)a.Q[K < 2 ? K + 1 : 2] + t.cw0, t.stepw, t.offt);
        if (NEED_L && K < 2) col_load<false>(lm, (const cpx<double> *)a.lam[K < 2 ? K + 1 : 2] + t.state0, t.steps, t.offs);
        if (t.live) {
            if (EH) col_store<false>(ac, (cpx<double> *)a.acc[K] + t.state0, t.steps, t.offs);
            if (MODE == ADJ_S0) col_store<false>(gn[K], (cpx<double> *)a.lam[K] + t.state0, t.steps, t.offs);
            else if (!FUSE) col_store<false>(gn[K], (cpx<double> *)a.lg[K] + t.state0, t.steps, t.offs);
        }
        if (NEED_A && K < 2) col_load<false>(ac, (const cpx<double> *)a.acc[K < 2 ? K + 1 : 2] + t.state0, t.steps, t.offs);
        pin_memory_order();
    }
    if constexpr (FUSE) xsym_columns<NT>(g, t, x, tw, a.S, gn);
}

template <typename T, int LL>
hipError_t xinv_sym_len(const XsymArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    hipLaunchKernelGGL((k_xinv_sym<T, LL, CB>), dim3(x_grid(x_tiles(a.g, CB, false))), dim3(CB * (LL / 8)), 0, st, a);
    return hipGetLastError();
}

template <typename T, int MM>
hipError_t z_adj_len(const ZArgs &a, hipStream_t st)
{
    const dim3 grid = ZLines<MM, 4>::grid(a.g), grid1 = ZLines<MM, 1>::grid(a.g);
    const bool nt = stream_bytes((size_t)8 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    if (nt) hipLaunchKernelGGL((k_z_adj<T, MM, true, 4>), grid, dim3(256), 0, st, a);
    else if (z_small<MM>(a.g)) hipLaunchKernelGGL((k_z_adj<T, MM, false, 1>), grid1, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_z_adj<T, MM, false, 4>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL, int MODE, bool FUSE>
hipError_t xfwd_adj_launch(const XadjArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    const bool nt = stream_bytes((size_t)8 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    constexpr bool NT = FUSE && LL >= kStreamLength;
    const dim3 grid(x_grid(x_tiles(a.g, CB, false))), block(CB * (LL / 8));
    if (NT && nt) hipLaunchKernelGGL((k_xfwd_adj<T, LL, CB, MODE, FUSE, NT>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_xfwd_adj<T, LL, CB, MODE, FUSE, false>), grid, block, 0, st, a);
    return hipGetLastError();
}

// Only the last stage of a sweep and ADJ_RHS end without a next stage.
template <typename T, int LL>
hipError_t xfwd_adj_len(const XadjArgs &a, bool fuse, hipStream_t st)
{
    if (a.ap.mode == ADJ_RHS && !fuse) return xfwd_adj_launch<T, LL, ADJ_RHS, false>(a, st);
    if (a.ap.mode == ADJ_S0 && !fuse) return xfwd_adj_launch<T, LL, ADJ_S0, false>(a, st);
    if (!fuse) return hipErrorInvalidValue;
    switch (a.ap.mode) {
        case ADJ_S0: return xfwd_adj_launch<T, LL, ADJ_S0, true>(a, st);
        case ADJ_S1: return xfwd_adj_launch<T, LL, ADJ_S1, true>(a, st);
        case ADJ_S2: return xfwd_adj_launch<T, LL, ADJ_S2, true>(a, st);
        case ADJ_S3: return xfwd_adj_launch<T, LL, ADJ_S3, true>(a, st);
        default: return hipErrorInvalidValue;
    }
}

#define TG_ADJ_L(N, T, P)                                                     \
    P template hipError_t xinv_sym_len<T, N>(const XsymArgs &, hipStream_t); \
    P template hipError_t xfwd_adj_len<T, N>(const XadjArgs &, bool, hipStream_t);
#define TG_ADJ_M(N, T, P) P template hipError_t z_adj_len<T, N>(const ZArgs &, hipStream_t);

#if TG_LEN_UNIT == 0
TG_ALL_UNITS(TG_ADJ_L, TG_ADJ_M, extern)

template <typename T>
hipError_t launch_xinv_sym(const Grid &g, double *const *G, void *const *S, const void *twx, hipStream_t st)
{
    XsymArgs a{};
    for (int i = 0; i < 3; i++) a.G[i] = G[i];
    for (int i = 0; i < 5; i++) a.S[i] = S[i];
    a.tw = twx;
    a.g = g;
    TG_DISPATCH_L(T, g.nx, return (xinv_sym_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_z_adj(const Grid &g, void *const *S, void *const *Q, void *const *tape, const void *twm,
                        const void *twn, hipStream_t st)
{
    ZArgs a{};
    for (int i = 0; i < 5; i++) a.in[i] = S[i];
    for (int i = 0; i < 3; i++) {
        a.out[i] = Q[i];
        a.tape[i] = tape[i];
    }
    a.twm = twm;
    a.twn = twn;
    a.g = g;
    TG_DISPATCH_M(T, g.nz / 2, return (z_adj_len<T, MM>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_xfwd_adj(const Grid &g, const AdjParams &ap, void *const *Q, double *const *lam,
                           double *const *acc, double *const *lg, const void *twx, hipStream_t st,
                           void *const *S_next)
{
    XadjArgs a{};
    if (S_next && ap.mode == ADJ_RHS) return hipErrorInvalidValue;
    for (int i = 0; i < 5; i++) a.S[i] = S_next ? S_next[i] : nullptr;
    for (int i = 0; i < 3; i++) {
        a.Q[i] = Q[i];
        a.lam[i] = lam ? lam[i] : nullptr;
        a.acc[i] = acc ? acc[i] : nullptr;
        a.lg[i] = lg ? lg[i] : nullptr;
    }
    a.tw = twx;
    a.g = g;
    a.ap = ap;
    TG_DISPATCH_L(T, g.nx, return (xfwd_adj_len<T, LL>)(a, S_next != nullptr, st));
    return hipErrorInvalidValue;
}

#define TG_ADJ_INST(T)                                                                                           \
    template hipError_t launch_xinv_sym<T>(const Grid &, double *const *, void *const *, const void *, hipStream_t); \
    template hipError_t launch_z_adj<T>(const Grid &, void *const *, void *const *, void *const *, const void *,  \
                                        const void *, hipStream_t);                                              \
    template hipError_t launch_xfwd_adj<T>(const Grid &, const AdjParams &, void *const *, double *const *,       \
                                           double *const *, double *const *, const void *, hipStream_t,         \
                                           void *const *);

TG_ADJ_INST(double)
TG_ADJ_INST(float)
#else
TG_THIS_UNIT(TG_ADJ_L, TG_ADJ_M)
#endif  // TG_LEN_UNIT

}  // namespace tg
