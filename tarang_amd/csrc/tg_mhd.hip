// tg_mhd.hip -- MHD (Elsasser) stage kernels.
//
// The nonlinear term of MHD (compute_nlin_VF_MHD.cc:71-123) runs through the
// giver transform pipeline with u = Z- and w = Z+: the nine products
// Z-_j Z+_i give N+_i = sum_j d_j(Z-_j Z+_i) (giver form) and
// N-_j = sum_i d_i(Z+_i Z-_j) (transposed giver form).  The kernels here:
//   k_xinv_elsasser x-inverse of Z+ = D(u) + D(b), Z- = D(u) - D(b) (stage-1
//                   input)
//   k_mhd_combine   N_u = (N+ + N-)/2, N_b = (N+ - N-)/2 (MHD.cc:150-163)
//                   for Compute_nlin
//   k_x_mhd         the fused x pass of an RK stage: x-forward of the eight
//                   trace-shifted products, N+ and N- together, their combination as
//                   above, RHS_u = -P N_u, RHS_b = -N_b (Tadvance_functions.cc:
//                   262-270), the Lawson RK4 stage for u (nu) and b (eta)
//                   (RK_VF_MHD.cc:126-190), and the x-inverse of the next
//                   stage's Z+- (one read of the products per stage; stage 4
//                   leaves the next step's stage-1 input)
#include <type_traits>

#include "tg_device.h"
#include "tg_kernels.h"
#include "tg_pass.h"
#include "tg_mhd.h"

namespace tg {

struct MhdArgs {
    double *V[3], *W[3];        // u, b (FP64 state)
    Grid g;
};

// x-inverse of Z- = D(u) - D(b) and Z+ = D(u) + D(b) into U[0..2] and U[3..5]
// (stage-1 input, Compute_nlin), straight from the state: forming Z+- in
// fields of their own first took 2.7 + 3.3 ms at 512^3 FP32 transforms.
// patch: the kz = 0 and Nz/2 columns only (after the reality condition has
// rewritten them).
struct XelsArgs {
    const double *V[3], *W[3];
    void *U[6];
    const void *tw;
    Grid g;
    int patch;
};

template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xinv_elsasser(XelsArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, a.patch)) return;
    const ColTile<T, L, CB> t(g, tile, a.patch);
    const int j = t.j;
    cpx<double> u[8], b[8];
    col_load<false>(u, (const cpx<double> *)a.V[0] + t.state0, t.steps, t.offs);
    col_load<false>(b, (const cpx<double> *)a.W[0] + t.state0, t.steps, t.offs);
    for (int i = threadIdx.x; i < L; i += CB * TPL) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    const X x{lds + t.c};
    int zx0, zx1;
    dealias_rows(g, t.ly, t.lz, zx0, zx1);
    if (!t.live) { zx0 = 0; zx1 = L - 1; }
#pragma unroll
    for (int K = 0; K < 3; K++) {
        const int jh = hidden(j);
        cpx<T> zp[8], zm[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            if (lx >= zx0 && lx <= zx1) u[s] = b[s] = mk<double>(0, 0);
            zp[s] = cvt<T>(u[s] + b[s]);
            zm[s] = cvt<T>(u[s] - b[s]);
            settle(zp[s]);
            settle(zm[s]);
        }
        pin_memory_order();
        if (K < 2) {
            col_load<false>(u, (const cpx<double> *)a.V[K < 2 ? K + 1 : 2] + t.state0, t.steps, t.offs);
            col_load<false>(b, (const cpx<double> *)a.W[K < 2 ? K + 1 : 2] + t.state0, t.steps, t.offs);
        }
        fft_exchange<L, +1>(zm, x, tw, hidden(j));
        if (t.inside) col_store<false>(zm, (cpx<T> *)a.U[K] + t.cw0, t.stepw, t.offt);
        fft_exchange<L, +1>(zp, x, tw, hidden(j));
        if (t.inside) col_store<false>(zp, (cpx<T> *)a.U[3 + K] + t.cw0, t.stepw, t.offt);
        pin_memory_order();
    }
}

#if TG_LEN_UNIT == 0
__global__ void k_mhd_combine(MhdArgs a)
{
    const Grid &g = a.g;
    const size_t n = (size_t)g.nx * g.ny * g.nzc;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        for (int c = 0; c < 3; c++) {
            cpx<double> *pp = (cpx<double> *)a.V[c] + i, *mm = (cpx<double> *)a.W[c] + i;
            const cpx<double> p = *pp, m = *mm;
            *pp = 0.5 * (p + m);
            *mm = 0.5 * (p - m);
        }
}

#endif  // TG_LEN_UNIT == 0

// ---------------------------------------------------------------------------
// Fused MHD x pass (stages 1-4).
// ---------------------------------------------------------------------------
// giver-form product order of the eight trace-shifted products (P_xx - P_zz,
// P_yy - P_zz, the off-diagonal ones; P_zz itself is not formed): the stage
// uses N_u = (N+ + N-)/2 only projected, and the shift changes N+ and N- by
// the same gradient -i K P_zz, so N_b = (N+ - N-)/2 is unchanged
constexpr int mhd_index(int pi)
{
    constexpr int order[8] = {0, 4, 3, 1, 7, 5, 2, 6};
    return order[pi];
}

// As k_x_nlin: columns in registers in transform order, the next tile in
// flight, products unrolled, code per stage, values settled where they are
// formed.  The six sums take 192 registers in FP64: blocks of 512 threads spill
// about 120 of them a lane, which costs less than rows of half the width in
// blocks of 256 (512 registers a thread): a step at 320 x 320 x 240 16 ms against
// 29, 512 x 256 x 512 33 against 34, 1024 x 256 x 512 82 against 89.
// The lambdas are inlined by attribute: left to the compiler, the x-inverse was a
// function at 240, 384 and 480 points and from 640 on, its columns passed through
// memory and its caller's registers saved around each call (1024 x 256 x 512: 23 ms a
// launch and 129 a step, now 11 and 82).
// 512^3 FP32, per launch: 11.0 ms, now 5.1 in stage 1, 5.9 in stages 2 and 3
// (4.8 TB/s), 7.1 in stage 4.
template <typename T, int L, int CB, int ST, bool NT>
__global__ void __launch_bounds__(CB *(L / 8), CB * (L / 8) <= 256 ? 1 : 2) k_x_mhd(XmhdArgs a)
{
    constexpr int TPL = L / 8, NTH = CB * TPL;
    constexpr bool NTW = NT && CB * sizeof(cpx<T>) >= 128, NTA = NT && CB * sizeof(cpx<double>) >= 128;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    // the viscous factors of u and b at this thread's points: exp(-nu K^2
    // dt/2), in stage 4 exp(-nu K^2 dt)
    __shared__ double visc[2][8 * NTH];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, false)) return;
    const ColTile<T, L, CB> t(g, tile);
    const int j = t.j, ly = t.ly, lz = t.lz;
    const double Ky = kwave(ly, g.ny) * g.kf[1], Kz = lz * g.kf[2];
    const T sc = (T)a.scale;
    const T Kyt = (T)Ky, Kzt = (T)Kz;
    cpx<T> cur[8], alt[8];
    col_load<NTW>(cur, (const cpx<T> *)a.P[mhd_index(0)] + t.cw0, t.stepw, t.offt);
    for (int i = threadIdx.x; i < L; i += NTH) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    const X x{lds + t.c};

    // --- x-forward of the products P[3i+j] = FT[Z-_j Z+_i]: N+_i += i K_j q
    // (giver form), N-_j += i K_i q (transposed) ---
    cpx<T> Np[3][8], Nm[3][8];
#pragma unroll
    for (int s = 0; s < 8; s++) Np[0][s] = Np[1][s] = Np[2][s] = Nm[0][s] = Nm[1][s] = Nm[2][s] = mk<T>(0, 0);
    cpx<double> w[8];   // the state of u, then of b, of one component
    auto product = [&](auto pc, cpx<T> *v, cpx<T> *next) __attribute__((always_inline)) {
        constexpr int PI = decltype(pc)::value;
        constexpr int P = mhd_index(PI), I = P / 3, J = P % 3;
        pin_memory_order();
        if constexpr (PI + 1 < 8) col_load<NTW>(next, (const cpx<T> *)a.P[mhd_index(PI < 7 ? PI + 1 : 7)] + t.cw0, t.stepw, t.offt);
        else col_load<false>(w, (const cpx<double> *)a.V[0] + t.state0, t.steps, t.offs);
        pin_memory_order();
        const int jh = hidden(j);
        fft_exchange<L, -1>(v, x, tw, jh);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const T Kx = (T)(kwave(jh + TPL * s, g.nx) * g.kf[0]);
            const cpx<T> q = sc * v[s];
            const T Kj = J == 0 ? Kx : (J == 1 ? Kyt : Kzt);
            const T Ki = I == 0 ? Kx : (I == 1 ? Kyt : Kzt);
            Np[I][s] = Np[I][s] + mul_i(Kj, q);
            Nm[J][s] = Nm[J][s] + mul_i(Ki, q);
            settle(Np[I][s]);
            settle(Nm[J][s]);
        }
    };
    product(std::integral_constant<int, 0>{}, cur, alt);
    product(std::integral_constant<int, 1>{}, alt, cur);
    product(std::integral_constant<int, 2>{}, cur, alt);
    product(std::integral_constant<int, 3>{}, alt, cur);
    product(std::integral_constant<int, 4>{}, cur, alt);
    product(std::integral_constant<int, 5>{}, alt, cur);
    product(std::integral_constant<int, 6>{}, cur, alt);
    product(std::integral_constant<int, 7>{}, alt, cur);

    // --- N_u = (N+ + N-)/2, N_b = (N+ - N-)/2, pressure on N_u, right-hand
    // sides RHS_u = -(N_u + i K p), RHS_b = -N_b (in place: Np <- RHS_u,
    // Nm <- RHS_b) ---
    {
        const int jh = hidden(j);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            const double K0 = kwave(lx, g.nx) * g.kf[0];
            cpx<double> nu[3], nb[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const cpx<double> pp = cvt<double>(Np[k][s]), mm = cvt<double>(Nm[k][s]);
                nu[k] = 0.5 * (pp + mm);
                nb[k] = 0.5 * (pp - mm);
            }
            const double kxs = K0 * K0;
            const double ks = (kxs + Ky * Ky) + Kz * Kz;
            cpx<double> div = mul_i(K0, nu[0]);
            div = div + mul_i(Ky, nu[1]);
            div = div + mul_i(Kz, nu[2]);
            cpx<double> pr = mk<double>(0, 0);
            if (!(lx == 0 && ly == 0 && lz == 0)) pr = mk<double>(div.x / ks, div.y / ks);
            const double Kc[3] = {K0, Ky, Kz};
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const cpx<double> ru = nu[k] + mul_i(Kc[k], pr);
                Np[k][s] = cvt<T>(mk<double>(-ru.x, -ru.y));
                Nm[k][s] = cvt<T>(mk<double>(-nb[k].x, -nb[k].y));
                settle(Np[k][s]);
                settle(Nm[k][s]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // --- Lawson stage for u (nu) and b (eta), next Z+- ---
    int zx0, zx1;
    dealias_rows(g, ly, lz, zx0, zx1);
    if (!t.live) { zx0 = 0; zx1 = L - 1; }
    auto ksq = [&](int lx) {
        const double K0 = kwave(lx, g.nx) * g.kf[0];
        return (K0 * K0 + Ky * Ky) + Kz * Kz;
    };
    {
        const int jh = hidden(j);
#pragma unroll 2
        for (int s = 0; s < 8; s++) {
            const double ks = ksq(jh + TPL * s);
            visc[0][s * NTH + threadIdx.x] = exp((ST == 4 ? a.f1_u : a.fh_u) * ks);
            visc[1][s * NTH + threadIdx.x] = exp((ST == 4 ? a.f1_b : a.fh_b) * ks);
        }
    }
    cpx<double> ac[8];
    if (ST >= 2) col_load<NTA>(ac, (const cpx<double> *)a.accV[0] + t.cw0, t.stepw, t.offw);
    double chk = 0.0;   // stage 4: NaN after a non-finite value
    // the accumulator, or the new state
    auto put = [&](double *acc, double *state) __attribute__((always_inline)) {
        if (ST == 4) {
            if (t.live) col_store<false>(ac, (cpx<double> *)state + t.state0, t.steps, t.offs);
        } else if (t.inside) {
            col_store<NTA>(ac, (cpx<double> *)acc + t.cw0, t.stepw, t.offw);
        }
    };
    // x-inverse of the next stage input (stage 4: of the next step's
    // first stage, D(u) +- D(b) of the new state)
    auto inverse = [&](cpx<T> *z, void *u) __attribute__((always_inline)) {
        pin_memory_order();
        fft_exchange<L, +1>(z, x, tw, hidden(j));
        pin_memory_order();
        if (t.inside) col_store<NTW>(z, (cpx<T> *)u + t.cw0, t.stepw, t.offt);
    };
    // Z+ of component K - 1 is transformed while b of component K is
    // loaded, its Z- while u of component K + 1 is
    cpx<T> zp[8], zm[8], zl[8];
    auto comp = [&](auto kc) __attribute__((always_inline)) {
        constexpr int K = decltype(kc)::value;
        constexpr int K1 = K < 2 ? K + 1 : 2;
        cpx<double> un[8];
        {
            const int jh = hidden(j);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int lx = jh + TPL * s;
                const bool z = lx >= zx0 && lx <= zx1;
                if (ST == 1 && z) w[s] = mk<double>(0, 0);
                const double E1 = ST == 1 ? exp(a.f1_u * ksq(lx)) : 0.0;
                lawson<ST>(w[s], cvt<double>(Np[K][s]), visc[0][s * NTH + threadIdx.x], E1, a.dt, ac[s], un[s]);
                if (ST == 4) {
                    chk += 0.0 * un[s].x + 0.0 * un[s].y;
                    settle(chk);
                }
                if (z) un[s] = mk<double>(0, 0);
                settle(un[s]);
                settle(ac[s]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        pin_memory_order();
        col_load<false>(w, (const cpx<double> *)a.W[K] + t.state0, t.steps, t.offs);
        put(a.accV[K], a.V[K]);
        if (ST >= 2) col_load<NTA>(ac, (const cpx<double> *)a.accW[K] + t.cw0, t.stepw, t.offw);
        if (K > 0) {
            inverse(zp, a.U[3 + (K > 0 ? K - 1 : 0)]);
#pragma unroll
            for (int s = 0; s < 8; s++) zl[s] = zm[s];
        }
        {
            const int jh = hidden(j);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int lx = jh + TPL * s;
                const bool z = lx >= zx0 && lx <= zx1;
                if (ST == 1 && z) w[s] = mk<double>(0, 0);
                const double E1 = ST == 1 ? exp(a.f1_b * ksq(lx)) : 0.0;
                cpx<double> bn;
                lawson<ST>(w[s], cvt<double>(Nm[K][s]), visc[1][s * NTH + threadIdx.x], E1, a.dt, ac[s], bn);
                if (ST == 4) {
                    chk += 0.0 * bn.x + 0.0 * bn.y;
                    settle(chk);
                }
                if (z) bn = mk<double>(0, 0);
                zp[s] = cvt<T>(un[s] + bn);
                zm[s] = cvt<T>(un[s] - bn);
                settle(zp[s]);
                settle(zm[s]);
                settle(ac[s]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        pin_memory_order();
        if (K < 2) col_load<false>(w, (const cpx<double> *)a.V[K1] + t.state0, t.steps, t.offs);
        put(a.accW[K], a.W[K]);
        if (ST >= 2 && K < 2) col_load<NTA>(ac, (const cpx<double> *)a.accV[K1] + t.cw0, t.stepw, t.offw);
        if (K > 0) inverse(zl, a.U[K > 0 ? K - 1 : 0]);
    };
    comp(std::integral_constant<int, 0>{});
    comp(std::integral_constant<int, 1>{});
    comp(std::integral_constant<int, 2>{});
    inverse(zp, a.U[5]);
    inverse(zm, a.U[2]);
    if (ST == 4 && chk != 0.0 && t.live && a.nonfinite) *a.nonfinite = 1;
}

template <typename T, int LL>
hipError_t x_mhd_len(const XmhdArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    const bool nt = stream_bytes((size_t)14 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    const dim3 grid(x_grid(x_tiles(a.g, CB, false))), block(CB * (LL / 8));
    auto go = [&](auto sc) {
        constexpr int ST = decltype(sc)::value;
        constexpr bool NT = LL >= kStreamLength;
        if (NT && nt) hipLaunchKernelGGL((k_x_mhd<T, LL, CB, ST, NT>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k_x_mhd<T, LL, CB, ST, false>), grid, block, 0, st, a);
    };
    if (a.stage == 1) go(std::integral_constant<int, 1>{});
    else if (a.stage == 2) go(std::integral_constant<int, 2>{});
    else if (a.stage == 3) go(std::integral_constant<int, 3>{});
    else go(std::integral_constant<int, 4>{});
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t xinv_elsasser_len(const XelsArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512);
    hipLaunchKernelGGL((k_xinv_elsasser<T, LL, CB>), dim3(x_grid(x_tiles(a.g, CB, a.patch))), dim3(CB * (LL / 8)), 0,
                       st, a);
    return hipGetLastError();
}

#define TG_MHD_L(N, T, P)                                                    \
    P template hipError_t x_mhd_len<T, N>(const XmhdArgs &, hipStream_t);   \
    P template hipError_t xinv_elsasser_len<T, N>(const XelsArgs &, hipStream_t);

#if TG_LEN_UNIT == 0
TG_ALL_UNITS(TG_MHD_L, TG_NO_LENGTHS, extern)

template <typename T>
hipError_t launch_x_mhd(const XmhdArgs &a, hipStream_t st)
{
    TG_DISPATCH_L(T, a.g.nx, return (x_mhd_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template hipError_t launch_x_mhd<double>(const XmhdArgs &, hipStream_t);
template hipError_t launch_x_mhd<float>(const XmhdArgs &, hipStream_t);

static MhdArgs mhd_args(const Grid &g, double *const *V, double *const *W)
{
    MhdArgs a{};
    for (int c = 0; c < 3; c++) {
        a.V[c] = V[c];
        a.W[c] = W[c];
    }
    a.g = g;
    return a;
}

template <typename T>
hipError_t launch_xinv_elsasser(const Grid &g, double *const *V, double *const *W, void *const *U, bool patch,
                                const void *twx, hipStream_t st)
{
    XelsArgs a{};
    for (int c = 0; c < 3; c++) {
        a.V[c] = V[c];
        a.W[c] = W[c];
        a.U[c] = U[c];
        a.U[3 + c] = U[3 + c];
    }
    a.tw = twx;
    a.g = g;
    a.patch = patch;
    TG_DISPATCH_L(T, g.nx, return (xinv_elsasser_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template hipError_t launch_xinv_elsasser<double>(const Grid &, double *const *, double *const *, void *const *, bool,
                                                 const void *, hipStream_t);
template hipError_t launch_xinv_elsasser<float>(const Grid &, double *const *, double *const *, void *const *, bool,
                                                const void *, hipStream_t);

hipError_t launch_mhd_combine(const Grid &g, double *const *NU, double *const *NW, hipStream_t st)
{
    MhdArgs a = mhd_args(g, NU, NW);
    hipLaunchKernelGGL(k_mhd_combine, dim3(4096), dim3(256), 0, st, a);
    return hipGetLastError();
}

#else
TG_THIS_UNIT(TG_MHD_L, TG_NO_LENGTHS)
#endif  // TG_LEN_UNIT

}  // namespace tg
