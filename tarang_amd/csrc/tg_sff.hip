// tg_sff.hip -- SFF basis kernels (sin/cos along x) and the Rayleigh-Benard
// stage pipeline on it.
//
// x transforms.  The reference's sin/cos transforms live in the absent fftk
// library; this build's convention (cell-centred samples x_j = (j+1/2)L/N,
// f_j = sum_m w_m A_m phi_m(x_j), w_0 = 1, w_m = 2, phi = sin or cos of
// m pi x / L; forward A = DCT-II/(2N), or the DST-II/(2N) shifted so that
// index m holds sin(m pi x / L), A_0 = 0) follows the reference's SFF energy
// (SFF_pencil_energy.cc:88-104) and x-derivative (SFF_pencil_tr.cc:84-105)
// formulas.  Each line transform is one complex FFT of length N
// (Makhoul's reordering): v_n = f_{2n}, v_{N-1-n} = f_{2n+1};
//   cosine forward   2N A_k = W^k V_k + W^-k V_{N-k},   V = FFT(v)
//   sine forward     the cosine transform of (-1)^j f_j, read backwards:
//                    2N A_m = i (W^m V_m - W^-m V_{N-m}), A_0 = 0
//   cosine inverse   V_k = W^-k (A_k - i A_{N-k}), v = IFFT(V) (unscaled)
//   sine inverse     V_k = W^-k (A_{N-k} - i A_k), V_0 = 0, then (-1)^j
// with W = exp(-i pi / (2N)) (table twq) and the (k, N-k) pairs exchanged
// through LDS.  A thread holds k = j + TPL*s (s < 8), and every pass forms
// W^k = W^j W^(TPL s) from those TPL + 8 table entries (QuarterTw), so all
// sin/cos passes round alike and keep only 8 + TPL entries in LDS.  A thread's
// samples are loaded and stored at their Makhoul positions directly (rows 2j
// apart, from both ends), so the reordering costs no pass through LDS.  Along y and z the FFF passes are reused.
#include <type_traits>

#include "tg_device.h"
#include "tg_pass.h"
#include "tg_sff.h"

namespace tg {

template <typename T>
__device__ __forceinline__ cpx<T> times_i(cpx<T> z) { return mk<T>(-z.y, z.x); }

// Post-twiddle W^(j + TPL*s) for the sin/cos line transforms.
template <typename T>
struct QuarterTw {
    const cpx<T> *lo;  // W^j, j < TPL
    const cpx<T> *hi;  // W^(TPL s), s < 8
    __device__ __forceinline__ cpx<T> operator()(int j, int s) const { return lo[j] * hi[s]; }
};

// Forward transform of a column: v[s] holds the sample at Makhoul position
// j + TPL*s; on return 2N A_k at k = j + TPL*s.
template <int L, typename X, typename T>
__device__ __forceinline__ void sc_forward(cpx<T> *v, const X &x, const cpx<T> *tw, const QuarterTw<T> &twq, int j, bool sine)
{
    constexpr int TPL = L / 8;
    if (sine) {
#pragma unroll
        for (int s = 4; s < 8; s++) v[s] = mk<T>(-v[s].x, -v[s].y);
    }
    fft_exchange<L, -1>(v, x, tw, j);
#pragma unroll
    for (int s = 0; s < 8; s++) x.w(j + TPL * s) = v[s];
    x.publish();
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = j + TPL * s;
        const cpx<T> vn = x.r(k == 0 ? 0 : L - k);
        const cpx<T> w = twq(j, s);
        const cpx<T> p = w * v[s];
        const cpx<T> q = conj(w) * vn;
        if (!sine) v[s] = p + q;
        else v[s] = k == 0 ? mk<T>(0, 0) : times_i(p - q);
    }
    x.release();
}

// Inverse: A_k in v[s] (k = j + TPL*s); on return the sample at Makhoul
// position j + TPL*s.
template <int L, typename X, typename T>
__device__ __forceinline__ void sc_inverse(cpx<T> *v, const X &x, const cpx<T> *tw, const QuarterTw<T> &twq, int j, bool sine)
{
    constexpr int TPL = L / 8;
#pragma unroll
    for (int s = 0; s < 8; s++) x.w(j + TPL * s) = v[s];
    x.publish();
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = j + TPL * s;
        cpx<T> an = x.r(k == 0 ? 0 : L - k);
        if (k == 0) an = mk<T>(0, 0);
        const cpx<T> ak = v[s];
        // component-wise selects (a select of the two values as objects keeps
        // v[] out of registers)
        const cpx<T> p = mk<T>(sine ? an.x : ak.x, sine ? an.y : ak.y);
        const cpx<T> q = mk<T>(sine ? ak.x : an.x, sine ? ak.y : an.y);
        cpx<T> z = conj(twq(j, s)) * mk<T>(p.x + q.y, p.y - q.x);  // W^-k (p - i q)
        if (sine && k == 0) z = mk<T>(0, 0);
        v[s] = z;
    }
    x.release();
    fft_exchange<L, +1>(v, x, tw, j);
    if (sine) {
#pragma unroll
        for (int s = 4; s < 8; s++) v[s] = mk<T>(-v[s].x, -v[s].y);
    }
}

// A column tile whose T work fields are read and written in Makhoul order:
// position n = j + TPL s holds sample 2n (s < 4: row 2j of rows 2 TPL s on) or
// 2(N - n) - 1 (row 2 TPL - 1 - 2j of rows 2 TPL (7 - s) on).  Byte offsets
// below a quarter of a field.
template <typename T, int L, int CB>
struct ScTile : ColTile<T, L, CB> {
    uint32_t even, odd;
    __device__ __forceinline__ ScTile(const Grid &g, int tile, bool patch = false) : ColTile<T, L, CB>(g, tile, patch)
    {
        const uint32_t row = (uint32_t)(g.ny * g.nzp) * (uint32_t)sizeof(cpx<T>);
        const uint32_t col = this->offt - this->j * row;
        even = 2 * this->j * row + col;
        odd = (2 * ColTile<T, L, CB>::TPL - 1 - 2 * this->j) * row + col;
    }
    template <bool NT>
    __device__ __forceinline__ void load(cpx<T> *v, const void *f) const
    {
        typedef __attribute__((address_space(1))) const vec2<T> gvec;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const cpx<T> *p = (const cpx<T> *)f + this->cw0 + 2 * (s < 4 ? s : 7 - s) * this->stepw;
            gvec *q = (gvec *)(uniform_address(p) + (s < 4 ? even : odd));
            vec2<T> x;
            if constexpr (NT) x = __builtin_nontemporal_load(q);
            else x = *q;
            v[s] = mk<T>(x.x, x.y);
        }
    }
    template <bool NT>
    __device__ __forceinline__ void store(const cpx<T> *v, void *f) const
    {
        typedef __attribute__((address_space(1))) vec2<T> gvec;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            cpx<T> *p = (cpx<T> *)f + this->cw0 + 2 * (s < 4 ? s : 7 - s) * this->stepw;
            gvec *q = (gvec *)(uniform_address(p) + (s < 4 ? even : odd));
            vec2<T> x;
            x.x = v[s].x;
            x.y = v[s].y;
            if constexpr (NT) __builtin_nontemporal_store(x, q);
            else *q = x;
        }
    }
};

// The twiddles of a sin/cos x kernel in LDS (L + L/8 + 8 entries).
template <typename T, int L>
struct ScTwiddles {
    const cpx<T> *tw;
    QuarterTw<T> twq;
    // all threads of the block; ends in a barrier
    __device__ __forceinline__ ScTwiddles(cpx<T> *lds, const void *twx, const void *q) : tw(lds), twq{lds + L, lds + L + L / 8}
    {
        constexpr int TPL = L / 8;
        for (int i = threadIdx.x; i < L; i += blockDim.x) lds[i] = ((const cpx<T> *)twx)[i];
        for (int i = threadIdx.x; i < TPL; i += blockDim.x) lds[L + i] = ((const cpx<T> *)q)[i];
        if (threadIdx.x < 8) lds[L + TPL + threadIdx.x] = ((const cpx<T> *)q)[TPL * threadIdx.x];
        lds_barrier();
    }
};

// ---------------------------------------------------------------------------
// Plain x passes (tg_forward / tg_inverse, stage-1 inputs, reality patches)
// ---------------------------------------------------------------------------
struct XscArgs {
    double *V[4];
    void *U[4];
    const void *tw, *twq;
    Grid g;
    int ncomp, parity, flags;
    double scale;
};

template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xinv_sc(XscArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> ldw[L + TPL + 8];
    const Grid &g = a.g;
    const bool patch = (a.flags & 4) != 0;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, patch)) return;
    const ScTile<T, L, CB> t(g, tile, patch);
    const int j = t.j;
    cpx<double> d[8];
    col_load<false>(d, (const cpx<double> *)a.V[0] + t.state0, t.steps, t.offs);
    const ScTwiddles<T, L> tw(ldw, a.tw, a.twq);
    const X x{lds + t.c};
    int zx0 = 1, zx1 = 0;
    if (a.flags & 1) dealias_rows(g, t.ly, t.lz, zx0, zx1);
    if (!t.live) { zx0 = 0; zx1 = L - 1; }
    const double w = (a.flags & 8) ? 0.5 : 1.0;   // a_k = 2 A_k of Chebyshev coefficients, k > 0
#pragma unroll 1
    for (int comp = 0; comp < a.ncomp; comp++) {
        cpx<T> v[8];
        const int jh = hidden(j);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            v[s] = lx >= zx0 && lx <= zx1 ? mk<T>(0, 0) : cvt<T>(lx > 0 ? w * d[s] : d[s]);
            settle(v[s]);
        }
        pin_memory_order();
        if (comp + 1 < a.ncomp) col_load<false>(d, (const cpx<double> *)a.V[comp + 1] + t.state0, t.steps, t.offs);
        pin_memory_order();
        sc_inverse<L>(v, x, tw.tw, tw.twq, jh, ((a.parity >> comp) & 1) != 0);
        pin_memory_order();
        if (t.inside) t.template store<false>(v, a.U[comp]);
    }
}

template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xfwd_sc(XscArgs a)
{
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> ldw[L + L / 8 + 8];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(a.g, CB, false)) return;
    const ScTile<T, L, CB> t(a.g, tile);
    cpx<T> v[8];
    t.template load<false>(v, a.U[0]);
    const ScTwiddles<T, L> tw(ldw, a.tw, a.twq);
    const X x{lds + t.c};
#pragma unroll 1
    for (int comp = 0; comp < a.ncomp; comp++) {
        sc_forward<L>(v, x, tw.tw, tw.twq, hidden(t.j), ((a.parity >> comp) & 1) != 0);
        cpx<double> o[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            o[s] = a.scale * cvt<double>(v[s]);
            if ((a.flags & 8) && t.j + (L / 8) * s > 0) o[s] = 2.0 * o[s];
        }
        pin_memory_order();
        if (comp + 1 < a.ncomp) t.template load<false>(v, a.U[comp + 1]);
        pin_memory_order();
        if (t.live) col_store<false>(o, (cpx<double> *)a.V[comp] + t.state0, t.steps, t.offs);
    }
}

// ---------------------------------------------------------------------------
// x pass of the Chebyshev basis' nonlinear term
// ---------------------------------------------------------------------------
struct XchArgs {
    void *P[6];
    double *N[3], *div;
    const void *tw, *twq;
    Grid g;
    double scale;
};

// Chebyshev derivative of a column, a_k in v (k = j + TPL s) in, b_k out:
// c_k b_k = b_{k+2} + 2 (k+1) a_{k+1}, i.e. sums of 2 p a_p over p > k of the
// other parity.  Each thread sums 8 consecutive k and takes the sums of the
// chunks above from LDS (tot: 2 TPL CB entries).
template <int L, int CB, typename X>
__device__ __forceinline__ void cheb_deriv_column(cpx<double> *v, const X &x, cpx<double> *tot, int c, int j, double kf)
{
    constexpr int TPL = L / 8;
#pragma unroll
    for (int s = 0; s < 8; s++) x.w(j + TPL * s) = (2.0 * (j + TPL * s)) * v[s];
    x.publish();
    cpx<double> e = mk<double>(0, 0), o = e;   // sums over even and odd p
#pragma unroll
    for (int i = 0; i < 8; i++) {
        v[i] = x.r(8 * j + i);
        if (i % 2) o = o + v[i];
        else e = e + v[i];
    }
    tot[(2 * j) * CB + c] = e;
    tot[(2 * j + 1) * CB + c] = o;
    x.release();
    e = o = mk<double>(0, 0);
    for (int q = TPL - 1; q > j; q--) {
        e = e + tot[(2 * q) * CB + c];
        o = o + tot[(2 * q + 1) * CB + c];
    }
#pragma unroll
    for (int i = 7; i >= 0; i--) {
        cpx<double> b = i % 2 ? e : o;
        if (i % 2) o = o + v[i];
        else e = e + v[i];
        if (i == 0 && j == 0) b = 0.5 * b;
        x.w(8 * j + i) = kf * b;
    }
    x.publish();
#pragma unroll
    for (int s = 0; s < 8; s++) v[s] = x.r(j + TPL * s);
    x.release();
}

// One pass over the six products: with the transforms field by field and the
// products, derivatives and sums in kernels of their own, the nonlinear term
// took 56 launches, now five (105 us at 64 x 128 x 128, this kernel 35).
template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xfwd_chff(XchArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> ldw[L + TPL + 8];
    __shared__ cpx<T> tot[2 * TPL * CB];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, false)) return;
    const ScTile<T, L, CB> t(g, tile);
    const int j = t.j;
    const double Ky = kwave(t.ly, g.ny) * g.kf[1], Kz = t.lz * g.kf[2];
    cpx<T> v[8], next[8];
    t.template load<false>(next, a.P[0]);
    const ScTwiddles<T, L> tw(ldw, a.tw, a.twq);
    const X x{lds + t.c};
    cpx<T> N[3][8];
    // product P of axes A and B: N_A += d_B, N_B += d_A; the next one's load is
    // in flight behind the transform
    auto product = [&](auto pc, auto nc) {
        constexpr int P = decltype(pc)::value, PN = decltype(nc)::value;
        constexpr int A = P < 3 ? P : P - 3, B = P < 3 ? P : (P - 2) % 3;
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = next[s];
        pin_memory_order();
        if (PN >= 0) t.template load<false>(next, a.P[PN < 0 ? 0 : PN]);
        pin_memory_order();
        sc_forward<L>(v, x, tw.tw, tw.twq, j, false);
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = (j + TPL * s > 0 ? 2.0 * a.scale : a.scale) * v[s];
        // d_y and d_z first: the x derivative replaces v
        auto add = [&](auto dst, auto dir) {
            constexpr int D = decltype(dst)::value, R = decltype(dir)::value;
            if constexpr (R > 0) {
#pragma unroll
                for (int s = 0; s < 8; s++) N[D][s] = N[D][s] + mul_i(R == 1 ? Ky : Kz, v[s]);
            }
        };
        add(std::integral_constant<int, A>{}, std::integral_constant<int, B>{});
        if constexpr (A != B) add(std::integral_constant<int, B>{}, std::integral_constant<int, A>{});
        if constexpr (A == 0 || B == 0) {
            constexpr int D = A == 0 ? B : A;
            cheb_deriv_column<L, CB>(v, x, tot, t.c, j, g.kf[0]);
#pragma unroll
            for (int s = 0; s < 8; s++) N[D][s] = N[D][s] + v[s];
        }
    };
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int s = 0; s < 8; s++) N[i][s] = mk<T>(0, 0);
    product(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
    product(std::integral_constant<int, 3>{}, std::integral_constant<int, 5>{});
    product(std::integral_constant<int, 5>{}, std::integral_constant<int, 1>{});
    product(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
    product(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
    product(std::integral_constant<int, 2>{}, std::integral_constant<int, -1>{});
    if (t.live) {
#pragma unroll
        for (int i = 0; i < 3; i++) col_store<false>(N[i], (cpx<double> *)a.N[i] + t.state0, t.steps, t.offs);
    }
    if (a.div) {
        cheb_deriv_column<L, CB>(N[0], x, tot, t.c, j, g.kf[0]);
#pragma unroll
        for (int s = 0; s < 8; s++) N[0][s] = N[0][s] + mul_i(Ky, N[1][s]) + mul_i(Kz, N[2][s]);
        if (t.live) col_store<false>(N[0], (cpx<double> *)a.div + t.state0, t.steps, t.offs);
    }
}

// ---------------------------------------------------------------------------
// z pass of the RBC nonlinear terms (Compute_nlin_VxT, compute_diag_offdiag.cc
// :116-136, and the diag/offdiag products :47-112): the three velocity lines
// are loaded together, transformed once and held in registers for the six
// velocity products, then theta for the three u theta products; four c2r
// and nine r2c per line.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int rbc_pair(int ia, int ib)
{
    // out: 0 xx, 1 yy, 2 zz, 3 xy, 4 yz, 5 zx, 6 x theta, 7 y theta, 8 z theta
    if (ia == ib) return ia;
    if (ia == 0) return ib == 1 ? 3 : (ib == 2 ? 5 : 6);
    if (ia == 1) return ib == 2 ? 4 : 7;
    return 8;
}

// Two waves per SIMD also for FP64 512-point lines (a few spilled registers
// there; 19.3 ms per stage at 512x1024x1024 against 21.0 ms at one wave).
// SHIFT: an RK stage's velocity products are the trace-shifted u_x^2 - u_z^2,
// u_y^2 - u_z^2 and the off-diagonal ones (out[2], zz, not written): the stage
// uses the velocity term only projected, and the SFF projection removes the
// gradient of u_z^2 that the shift adds.
template <typename T, int M, bool SHIFT, bool NT, int W>
__global__ void __launch_bounds__(64 * W, 2) k_z_rbc(ZArgs a)
{
    constexpr int TPL = M / 8;
    constexpr int LPB = ZLines<M, W>::LPB;
    constexpr int LP = lpad_len(M);
    __shared__ cpx<T> lds[LPB * LP], ldw[2 * M];
    const ZLines<M, W> z(a.g);
    const int li = z.li, j = z.j;
    const size_t lsafe = z.safe;
    const bool valid = z.valid;
    cpx<T> *L = lds + li * LP;
    const size_t off = lsafe * a.g.nzp;
    cpx<T> u[3][8], xm[3];
#pragma unroll
    for (int c = 0; c < 3; c++) zline_load<T, M, NT>(u[c], xm[c], (const cpx<T> *)a.in[c] + off, j);
    const ZTwiddles<T, M> tw(ldw, a.twm, a.twn);
    if (z.spare) return;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        zline_c2r_from<T, M>(u[c], xm[c], L, tw, j);
        line_sync();
    }
    auto emit = [&](const cpx<T> *x, const cpx<T> *y, int o) {
        cpx<T> p[8];
#pragma unroll
        for (int s = 0; s < 8; s++) p[s] = mk<T>(x[s].x * y[s].x, x[s].y * y[s].y);
        zline_r2c_post<T, M, NT>(p, (cpx<T> *)a.out[o] + off, L, tw, j, valid, a.g.nzp - M);
    };
    if constexpr (SHIFT) {
        // the off-diagonal products first, then the shifted squares (u_z is
        // last used there)
        emit(u[0], u[1], rbc_pair(0, 1));
        emit(u[1], u[2], rbc_pair(1, 2));
        emit(u[0], u[2], rbc_pair(0, 2));
#pragma unroll
        for (int ia = 0; ia < 2; ia++) {
            cpx<T> p[8];
#pragma unroll
            for (int s = 0; s < 8; s++)
                p[s] = mk<T>(u[ia][s].x * u[ia][s].x - u[2][s].x * u[2][s].x,
                             u[ia][s].y * u[ia][s].y - u[2][s].y * u[2][s].y);
            zline_r2c_post<T, M, NT>(p, (cpx<T> *)a.out[ia] + off, L, tw, j, valid, a.g.nzp - M);
        }
    } else {
#pragma unroll
        for (int ia = 0; ia < 3; ia++)
#pragma unroll
            for (int ib = ia; ib < 3; ib++) emit(u[ia], u[ib], rbc_pair(ia, ib));
    }
    cpx<T> t[8];
    zline_c2r<T, M, NT>(t, (const cpx<T> *)a.in[3] + off, L, tw, j);
    line_sync();
#pragma unroll
    for (int ia = 0; ia < 3; ia++) emit(u[ia], t, rbc_pair(ia, 3));
}

// ---------------------------------------------------------------------------
// Fused x pass of an RBC stage.
// ---------------------------------------------------------------------------
struct XrbcArgs {
    void *P[9];
    double *V[4];
    double *acc[4];
    void *U[4];
    const double *f_in[2];
    double *f_out[2];
    double *out[4];
    const void *tw, *twq;
    Grid g;
    RbcParams rp;
};

// Terms of the nonlinear terms (SFF_pencil_tr.cc:77-151): the derivative of a
// transformed product q along axis D (x: +Kx q of an 'S' product, -Kx q of a
// 'C' one), added to n.  The term is settled before it is added: the passes
// round it on its own.
template <int D, bool SINE, typename T>
__device__ __forceinline__ void add_term(cpx<T> &n, T Kx, T Ky, T Kz, cpx<T> q)
{
    cpx<T> d;
    if constexpr (D == 0) d = SINE ? mk<T>(Kx * q.x, Kx * q.y) : mk<T>(-Kx * q.x, -Kx * q.y);
    else d = mul_i(D == 1 ? Ky : Kz, q);
    settle(d);
    n = n + d;
    settle(n);
}

// PHASE 0: temperature (N_T, its right-hand side, Lawson for theta, nu =
// kappa); PHASE 1: velocity.  The two launches of a stage touch disjoint data
// (the force inputs they read are the other field's, of this stage's input).
// ST: RK stage 1..4 (velocity products trace-shifted: xx - zz, yy - zz, zz not
// formed), 0 nonlinear terms or right-hand sides only (six products).
//
// Bound by HBM.  Columns go from memory to registers and back in transform
// order (the products and the next stage input in Makhoul order), the next
// load is in flight behind each transform, products and components are
// unrolled and each stage has its code: with the tiles staged through LDS the
// launches of a stage at 256 x 512 x 512 FP32 took 1.0 and 2.2 ms, now 0.85 and 1.83 (4.6 TB/s).
template <typename T, int L, int CB, int PHASE, int ST, bool NT>
__global__ void __launch_bounds__(CB *(L / 8), 2) k_x_rbc(XrbcArgs a)
{
    constexpr int TPL = L / 8, NTH = CB * TPL;
    constexpr bool NTW = NT && CB * sizeof(cpx<T>) >= 128, NTA = NT && CB * sizeof(cpx<double>) >= 128;
    constexpr int NC = PHASE == 0 ? 1 : 3;   // components of the phase
    constexpr int C0 = PHASE == 0 ? 3 : 0;   // the first one (u_x, u_y, u_z, theta)
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> ldw[L + TPL + 8];
    // the viscous factors at this thread's points: exp(-nu K^2 dt/2) (not in
    // stage 4), exp(-nu K^2 dt) (stages 1 and 4)
    __shared__ double visc[ST == 1 ? 2 : 1][ST > 0 ? 8 * NTH : 1];
    const Grid &g = a.g;
    const RbcParams &rp = a.rp;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, false)) return;
    const ScTile<T, L, CB> t(g, tile);
    const int j = t.j, ly = t.ly, lz = t.lz;
    const double Ky = kwave(ly, g.ny) * g.kf[1], Kz = lz * g.kf[2];
    const T Kyt = (T)Ky, Kzt = (T)Kz;
    const T sc = (T)rp.scale;
    const bool want_rhs = ST > 0 || rp.write_rhs;
    // the products of the phase: x theta C, y theta S, z theta S; xx C, yy C,
    // (zz C), xy S, yz C, zx S
    constexpr int NP = PHASE == 0 ? 3 : (ST > 0 ? 5 : 6);
    constexpr int first = PHASE == 0 ? 6 : 0;
    auto index = [](int q) { return PHASE == 1 && ST > 0 && q >= 2 ? q + 1 : first + q; };
    cpx<T> cur[8], alt[8];
    t.template load<NTW>(cur, a.P[first]);
    const ScTwiddles<T, L> tw(ldw, a.tw, a.twq);
    const X x{lds + t.c};
    cpx<T> N[NC][8];
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < 8; s++) N[k][s] = mk<T>(0, 0);
    cpx<double> w[8];
    auto product = [&](auto qc, cpx<T> *v, cpx<T> *next) {
        constexpr int Q = decltype(qc)::value;
        if constexpr (Q < NP) {
            constexpr int P = PHASE == 1 && ST > 0 && Q >= 2 ? Q + 1 : first + Q;
            constexpr bool SINE = P == 3 || P == 5 || P > 6;
            pin_memory_order();
            if constexpr (Q + 1 < NP) t.template load<NTW>(next, a.P[index(Q + 1)]);
            else if (want_rhs) col_load<false>(w, (const cpx<double> *)a.f_in[PHASE == 0 ? 1 : 0] + t.state0, t.steps, t.offs);
            pin_memory_order();
            const int jh = hidden(j);
            sc_forward<L>(v, x, tw.tw, tw.twq, jh, SINE);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const T Kx = (T)((jh + TPL * s) * g.kf[0]);
                const cpx<T> q = sc * v[s];
                if constexpr (P >= 6) {
                    add_term<P - 6, SINE>(N[0][s], Kx, Kyt, Kzt, q);
                } else if constexpr (P < 3) {
                    add_term<P, SINE>(N[P % NC][s], Kx, Kyt, Kzt, q);
                } else {
                    constexpr int A = P - 3, B = (P - 2) % 3;   // xy, yz, zx
                    add_term<B, SINE>(N[A % NC][s], Kx, Kyt, Kzt, q);
                    add_term<A, SINE>(N[B % NC][s], Kx, Kyt, Kzt, q);
                }
            }
        }
    };
    product(std::integral_constant<int, 0>{}, cur, alt);
    product(std::integral_constant<int, 1>{}, alt, cur);
    product(std::integral_constant<int, 2>{}, cur, alt);
    product(std::integral_constant<int, 3>{}, alt, cur);
    product(std::integral_constant<int, 4>{}, cur, alt);
    product(std::integral_constant<int, 5>{}, alt, cur);

    // --- right-hand sides (in place, negated) ---
    cpx<double> ac[8], v0[8];
    if (ST > 0) col_load<false>(v0, (const cpx<double> *)a.V[C0] + t.state0, t.steps, t.offs);
    pin_memory_order();
    cpx<double> rt[PHASE == 0 ? 8 : 1];   // RHS_T stays in FP64
    if constexpr (PHASE == 0) {
        // RHS_T = -(N_T - F_T), F_T = u_x of the stage input
#pragma unroll
        for (int s = 0; s < 8; s++) {
            rt[s] = cvt<double>(N[0][s]);
            if (want_rhs) {
                const cpx<double> n = rt[s] - w[s];
                rt[s] = mk<double>(-n.x, -n.y);
            }
            settle(rt[s]);
        }
    } else if (want_rhs) {
        // nlin -= F (F_x = theta of the stage input); p = div/K^2 with the SFF
        // divergence (+Kx on the 'S' x component); nlin += grad p ('C' parity:
        // -Kx p); negate (Compute_rhs_scalar)
        const int jh = hidden(j);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            const double Kx = lx * g.kf[0];
            cpx<double> n0 = cvt<double>(N[0][s]) - w[s];
            cpx<double> n1 = cvt<double>(N[1 % NC][s]), n2 = cvt<double>(N[2 % NC][s]);
            cpx<double> div = Kx * n0;
            div = div + mul_i(Ky, n1);
            div = div + mul_i(Kz, n2);
            const double ks = (Kx * Kx + Ky * Ky) + Kz * Kz;
            cpx<double> pr = mk<double>(0, 0);
            if (!(lx == 0 && ly == 0 && lz == 0)) pr = mk<double>(div.x / ks, div.y / ks);
            n0 = n0 + (-Kx) * pr;
            n1 = n1 + mul_i(Ky, pr);
            n2 = n2 + mul_i(Kz, pr);
            N[0][s] = cvt<T>(mk<double>(-n0.x, -n0.y));
            N[1 % NC][s] = cvt<T>(mk<double>(-n1.x, -n1.y));
            N[2 % NC][s] = cvt<T>(mk<double>(-n2.x, -n2.y));
            settle(N[0][s]);
            settle(N[1 % NC][s]);
            settle(N[2 % NC][s]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (ST == 0) {
#pragma unroll
        for (int k = 0; k < NC; k++) {
            cpx<double> o[8];
#pragma unroll
            for (int s = 0; s < 8; s++) o[s] = PHASE == 0 ? rt[PHASE == 0 ? s : 0] : cvt<double>(N[k][s]);
            if (t.live) col_store<false>(o, (cpx<double> *)a.out[C0 + k] + t.state0, t.steps, t.offs);
        }
    } else {
        // --- Lawson stage (RK_SF.cc:97-215 with Tadvance_functions.cc:298-324,
        // 566-570), next stage input ---
        int zx0, zx1;
        dealias_rows(g, ly, lz, zx0, zx1);
        if (!t.live) { zx0 = 0; zx1 = L - 1; }
        {
            const int jh = hidden(j);
            const double fh = PHASE == 0 ? rp.fh_t : rp.fh_u, f1 = PHASE == 0 ? rp.f1_t : rp.f1_u;
#pragma unroll 2
            for (int s = 0; s < 8; s++) {
                const double Kx = (jh + TPL * s) * g.kf[0];
                const double ks = (Kx * Kx + Ky * Ky) + Kz * Kz;
                visc[0][s * NTH + threadIdx.x] = exp((ST == 4 ? f1 : fh) * ks);
                if (ST == 1) visc[ST == 1][s * NTH + threadIdx.x] = exp(f1 * ks);
            }
        }
        if (ST >= 2) col_load<NTA>(ac, (const cpx<double> *)a.acc[C0] + t.cw0, t.stepw, t.offw);
        double chk = 0.0;   // stage 4: NaN after a non-finite value
        auto comp = [&](auto kc) {
            constexpr int K = decltype(kc)::value;
            constexpr int C = C0 + K;
            constexpr bool FORCE = ST < 4 && (C == 0 || C == 3);   // feeds the next stage's force
            cpx<T> v[8];
            {
                const int jh = hidden(j);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const int lx = jh + TPL * s;
                    const bool z = lx >= zx0 && lx <= zx1;
                    if (ST == 1 && z) v0[s] = mk<double>(0, 0);
                    const double E = visc[0][s * NTH + threadIdx.x];
                    const double E1 = ST == 1 ? visc[ST == 1][s * NTH + threadIdx.x] : 0.0;
                    cpx<double> vn;
                    lawson<ST>(v0[s], PHASE == 0 ? rt[PHASE == 0 ? s : 0] : cvt<double>(N[K][s]), E, E1, rp.dt, ac[s], vn);
                    if (ST == 4) {
                        chk += 0.0 * vn.x + 0.0 * vn.y;
                        settle(chk);
                    }
                    // the undealiased value is this field's share of the next force
                    if (FORCE) v0[s] = vn;
                    v[s] = z ? mk<T>(0, 0) : cvt<T>(vn);
                    settle(v[s]);
                    settle(ac[s]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            pin_memory_order();
            if (FORCE && t.live)
                col_store<false>(v0, (cpx<double> *)a.f_out[PHASE == 0 ? 0 : 1] + t.state0, t.steps, t.offs);
            if (K + 1 < NC) col_load<false>(v0, (const cpx<double> *)a.V[K + 1 < NC ? C + 1 : C] + t.state0, t.steps, t.offs);
            if (ST == 4) {
                if (t.live) col_store<false>(ac, (cpx<double> *)a.V[C] + t.state0, t.steps, t.offs);
            } else if (t.inside) {
                col_store<NTA>(ac, (cpx<double> *)a.acc[C] + t.cw0, t.stepw, t.offw);
            }
            if (ST >= 2 && K + 1 < NC)
                col_load<NTA>(ac, (const cpx<double> *)a.acc[K + 1 < NC ? C + 1 : C] + t.cw0, t.stepw, t.offw);
            pin_memory_order();
            sc_inverse<L>(v, x, tw.tw, tw.twq, hidden(j), C == 0 || C == 3);
            pin_memory_order();
            if (t.inside) t.template store<NTW>(v, a.U[C]);
        };
        comp(std::integral_constant<int, 0>{});
        if constexpr (NC > 1) {
            comp(std::integral_constant<int, (NC > 1 ? 1 : 0)>{});
            comp(std::integral_constant<int, (NC > 2 ? 2 : 0)>{});
        }
        if (ST == 4 && chk != 0.0 && t.live && rp.nonfinite) *rp.nonfinite = 1;
    }
}

// ---------------------------------------------------------------------------
// Reality conditions on SFF fields
// ---------------------------------------------------------------------------
struct SffPlaneArgs {
    double *V[4];
    Grid g;
    int ncomp, mode;
};

#if TG_LEN_UNIT == 0
__global__ void k_sff_reality(SffPlaneArgs a)
{
    const Grid &g = a.g;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.nx * g.ny) return;
    const int lx = i / g.ny, ly = i % g.ny;
    const int ky = kwave(ly, g.ny);
    for (int comp = 0; comp < a.ncomp; comp++) {
        cpx<double> *A = (cpx<double> *)a.V[comp];
        const size_t row = ((size_t)lx * g.ny + ly) * g.nzc;
        // A(lx, ky, 0) = conj A(lx, -ky, 0) for -Ny/2 < ky < 0 reads a
        // ky > 0 row, which this kernel never writes; ky = 0 conjugates in place
        if (a.mode == 1 && ky <= 0) {
            const cpx<double> src = A[((size_t)lx * g.ny + (-ky)) * g.nzc];
            A[row] = conj(src);
        }
        A[row + g.nzc - 1] = mk<double>(0, 0);
    }
}

#endif  // TG_LEN_UNIT == 0

// ---------------------------------------------------------------------------
// Per-length launch functions and launchers
// ---------------------------------------------------------------------------
template <typename T, int LL>
hipError_t xinv_sc_len(const XscArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    hipLaunchKernelGGL((k_xinv_sc<T, LL, CB>), dim3(x_grid(x_tiles(a.g, CB, (a.flags & 4) != 0))),
                       dim3(CB * (LL / 8)), 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t xfwd_sc_len(const XscArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    hipLaunchKernelGGL((k_xfwd_sc<T, LL, CB>), dim3(x_grid(x_tiles(a.g, CB, false))), dim3(CB * (LL / 8)), 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t xfwd_chff_len(const XchArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    if constexpr (sizeof(T) == 8)
        hipLaunchKernelGGL((k_xfwd_chff<T, LL, CB>), dim3(x_grid(x_tiles(a.g, CB, false))), dim3(CB * (LL / 8)), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <typename T, int MM>
hipError_t z_rbc_len(const ZArgs &a, hipStream_t st)
{
    const dim3 grid = ZLines<MM, 4>::grid(a.g), grid1 = ZLines<MM, 1>::grid(a.g);
    const bool nt = stream_bytes((size_t)12 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    if (a.ncomp != 8) hipLaunchKernelGGL((k_z_rbc<T, MM, false, false, 4>), grid, dim3(256), 0, st, a);
    else if (nt) hipLaunchKernelGGL((k_z_rbc<T, MM, true, true, 4>), grid, dim3(256), 0, st, a);
    else if (z_small<MM>(a.g)) hipLaunchKernelGGL((k_z_rbc<T, MM, true, false, 1>), grid1, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_z_rbc<T, MM, true, false, 4>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL, int ST>
hipError_t x_rbc_launch(const XrbcArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    const bool nt = stream_bytes((size_t)12 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    constexpr bool NT = ST > 0 && LL >= kStreamLength;
    const dim3 grid(x_grid(x_tiles(a.g, CB, false))), block(CB * (LL / 8));
    if (NT && nt) {
        hipLaunchKernelGGL((k_x_rbc<T, LL, CB, 0, ST, NT>), grid, block, 0, st, a);
        hipLaunchKernelGGL((k_x_rbc<T, LL, CB, 1, ST, NT>), grid, block, 0, st, a);
    } else {
        hipLaunchKernelGGL((k_x_rbc<T, LL, CB, 0, ST, false>), grid, block, 0, st, a);
        hipLaunchKernelGGL((k_x_rbc<T, LL, CB, 1, ST, false>), grid, block, 0, st, a);
    }
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t x_rbc_len(const XrbcArgs &a, hipStream_t st)
{
    switch (a.rp.stage) {
        case 1: return x_rbc_launch<T, LL, 1>(a, st);
        case 2: return x_rbc_launch<T, LL, 2>(a, st);
        case 3: return x_rbc_launch<T, LL, 3>(a, st);
        case 4: return x_rbc_launch<T, LL, 4>(a, st);
        default: return x_rbc_launch<T, LL, 0>(a, st);
    }
}

#define TG_SFF_L(N, T, P)                                                   \
    P template hipError_t xinv_sc_len<T, N>(const XscArgs &, hipStream_t); \
    P template hipError_t xfwd_sc_len<T, N>(const XscArgs &, hipStream_t); \
    P template hipError_t xfwd_chff_len<T, N>(const XchArgs &, hipStream_t); \
    P template hipError_t x_rbc_len<T, N>(const XrbcArgs &, hipStream_t);
#define TG_SFF_M(N, T, P) P template hipError_t z_rbc_len<T, N>(const ZArgs &, hipStream_t);

#if TG_LEN_UNIT == 0
TG_ALL_UNITS(TG_SFF_L, TG_SFF_M, extern)

template <typename T>
hipError_t launch_xinv_sc(const Grid &g, double *const *V, int ncomp, int parity, void *const *U, int flags,
                          const void *twx, const void *twq, hipStream_t st)
{
    XscArgs a{};
    for (int i = 0; i < ncomp; i++) {
        a.V[i] = V[i];
        a.U[i] = U[i];
    }
    a.tw = twx;
    a.twq = twq;
    a.g = g;
    a.ncomp = ncomp;
    a.parity = parity;
    a.flags = flags;
    TG_DISPATCH_L(T, g.nx, return (xinv_sc_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_xfwd_sc(const Grid &g, void *const *W, int ncomp, int parity, double *const *out, double scale,
                          const void *twx, const void *twq, hipStream_t st, int flags)
{
    XscArgs a{};
    a.flags = flags;
    for (int i = 0; i < ncomp; i++) {
        a.U[i] = W[i];
        a.V[i] = out[i];
    }
    a.tw = twx;
    a.twq = twq;
    a.g = g;
    a.ncomp = ncomp;
    a.parity = parity;
    a.scale = scale;
    TG_DISPATCH_L(T, g.nx, return (xfwd_sc_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

hipError_t launch_xfwd_chff(const Grid &g, void *const *P, double *const *N, double *div, double scale, const void *twx,
                            const void *twq, hipStream_t st)
{
    XchArgs a{};
    for (int i = 0; i < 6; i++) a.P[i] = P[i];
    for (int i = 0; i < 3; i++) a.N[i] = N[i];
    a.div = div;
    a.tw = twx;
    a.twq = twq;
    a.g = g;
    a.scale = scale;
    TG_DISPATCH_L(double, g.nx, return (xfwd_chff_len<double, LL>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_z_rbc(const Grid &g, void *const *U, void *const *P, const void *twm, const void *twn,
                        hipStream_t st, bool shift)
{
    ZArgs a{};
    a.ncomp = shift ? 8 : 9;
    for (int i = 0; i < 4; i++) a.in[i] = U[i];
    for (int i = 0; i < 9; i++) a.out[i] = P[i];
    a.twm = twm;
    a.twn = twn;
    a.g = g;
    TG_DISPATCH_M(T, g.nz / 2, return (z_rbc_len<T, MM>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_x_rbc(const Grid &g, const RbcParams &rp, void *const *P, double *const *V, double *const *acc,
                        void *const *U, const double *const *f_in, double *const *f_out, double *const *out,
                        const void *twx, const void *twq, hipStream_t st)
{
    XrbcArgs a{};
    for (int i = 0; i < 9; i++) a.P[i] = P[i];
    for (int i = 0; i < 4; i++) {
        a.V[i] = V ? V[i] : nullptr;
        a.acc[i] = acc ? acc[i] : nullptr;
        a.U[i] = U ? U[i] : nullptr;
        a.out[i] = out ? out[i] : nullptr;
    }
    for (int i = 0; i < 2; i++) {
        a.f_in[i] = f_in ? f_in[i] : nullptr;
        a.f_out[i] = f_out ? f_out[i] : nullptr;
    }
    a.tw = twx;
    a.twq = twq;
    a.g = g;
    a.rp = rp;
    TG_DISPATCH_L(T, g.nx, return (x_rbc_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

hipError_t launch_sff_reality(const Grid &g, double *const *V, int ncomp, int mode, hipStream_t st)
{
    SffPlaneArgs a{};
    for (int i = 0; i < ncomp; i++) a.V[i] = V[i];
    a.g = g;
    a.ncomp = ncomp;
    a.mode = mode;
    const int n = g.nx * g.ny;
    hipLaunchKernelGGL(k_sff_reality, dim3((n + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

#define TG_SFF_INST(T)                                                                                              \
    template hipError_t launch_xinv_sc<T>(const Grid &, double *const *, int, int, void *const *, int, const void *, \
                                          const void *, hipStream_t);                                               \
    template hipError_t launch_xfwd_sc<T>(const Grid &, void *const *, int, int, double *const *, double,           \
                                          const void *, const void *, hipStream_t, int);                            \
    template hipError_t launch_z_rbc<T>(const Grid &, void *const *, void *const *, const void *, const void *,     \
                                        hipStream_t, bool);                                                         \
    template hipError_t launch_x_rbc<T>(const Grid &, const RbcParams &, void *const *, double *const *,            \
                                        double *const *, void *const *, const double *const *, double *const *,     \
                                        double *const *, const void *, const void *, hipStream_t);

TG_SFF_INST(double)
TG_SFF_INST(float)
#else
TG_THIS_UNIT(TG_SFF_L, TG_SFF_M)
#endif  // TG_LEN_UNIT

}  // namespace tg
