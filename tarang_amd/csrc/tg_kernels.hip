// tg_kernels.hip -- gfx950 kernels of the pseudo-spectral FFF hot path.
//
// HBM layouts (all complex fields interleaved re/im):
//   spectral state  V(lx,ly,lz)        (Nx, Ny, Nz/2+1) FP64, kz fastest
//   work fields     W(x | ly | lz ...) (Nx, Ny, Nz/2+1) in the transform
//                   precision T; the same shape serves every intermediate
//                   of the 3D transform (x, y and z passes work in place on
//                   it, each pass finishing one axis).
//   real fields     R(x,y,z)           (Nx, Ny, Nz+2) FP64, z fastest.
//
// Passes:
//   x pass  tiles of all Nx rows x CB contiguous (ly,lz) columns, from memory to
//           registers and back in the transform's order (ColX); LDS carries the
//           exchanges between the radix passes, one line per TPL = Nx/8 threads.
//   y pass  tiles of all Ny rows x CB contiguous lz columns of one lx, likewise.
//   z pass  whole z-lines (contiguous), TPL = Nz/16 threads per line; a
//           real line of Nz points is packed as Nz/2 complex points.
#include <algorithm>
#include <type_traits>

#include "tg_device.h"
#include "tg_kernels.h"
#include "tg_pass.h"
#include "tg_aniso.h"
#include "tg_rand.h"

namespace tg {

// ---------------------------------------------------------------------------
// Column FFT along a strided axis (the y pass).
// ---------------------------------------------------------------------------
struct ColArgs {
    void *f[9];
    const void *tw;
    long long outer_stride;  // elements between tiles of different outer index
    long long row_stride;    // elements between consecutive rows (transform axis)
    int ncol;                // contiguous columns per row
    int nouter;
    int keep;                // CUT: rows |k| <= keep
};

// Bound by HBM (each field read and written once).  A thread's row segment and
// its share of the transform are the same points (ColX), so LDS carries only
// the exchanges between the radix passes; 512^3 FP64, per field: 476 us with
// the tile staged through LDS both ways, 381 us (5.7 TB/s, a copy's 6.2) with
// this layout, whole rows and non-temporal access.
// CUT: of the rows |k| > keep nothing is read (inverse) or written (forward).
template <typename T, int L, int DIR, int CB, bool NT, bool CUT>
__global__ void __launch_bounds__(CB *(L / 8)) k_colfft(ColArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    // xcd_tile: the column blocks of one outer index run in turn on one XCD,
    // so the rows' 128-byte lines that two blocks share (CB columns of fewer
    // than 128 bytes) are fetched into one L2
    const int nblk = (a.ncol + CB - 1) / CB;
    const int b = xcd_tile(blockIdx.x, gridDim.x);
    if (b >= a.nouter * nblk) return;
    const int outer = b / nblk;
    const int c0 = (b % nblk) * CB;
    const int c = threadIdx.x % CB, j = threadIdx.x / CB, col = c0 + c;
    // a column past the last one transforms the last one and is not stored
    cpx<T> *p = (cpx<T> *)a.f[blockIdx.y] + (size_t)outer * a.outer_stride + (size_t)j * a.row_stride +
                min(col, a.ncol - 1);
    const size_t step = (size_t)TPL * a.row_stride;
    cpx<T> v[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        v[s] = mk<T>(0, 0);
        if (!CUT || DIR < 0 || abs(kwave(j + TPL * s, L)) <= a.keep) v[s] = gload<NT>(p + s * step);
    }
    const X x{lds + c};
    fft_exchange<L, DIR>(v, x, (const cpx<T> *)a.tw, j);
    if (col < a.ncol) {
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (!CUT || DIR > 0 || abs(kwave(j + TPL * s, L)) <= a.keep) gstore<NT>(p + s * step, v[s]);
    }
}

// ---------------------------------------------------------------------------
// x-inverse of FP64 spectral fields into T work fields (first pass of the
// 3D inverse transform; stage-1 input of an RK4 step).
// ---------------------------------------------------------------------------
struct XinvArgs {
    double *V[3];
    void *U[3];
    double *slots;
    const void *tw;
    Grid g;
    Band b;
    int ncomp, flags;
    double r_lo, r_hi;  // flags & 8: keep only r_lo < K <= r_hi (Fill_array_shell)
    // flags & 16: ring r_lo < K <= r_hi, a_lo < theta <= a_hi (Fill_array_ring);
    // flags & 32: cylindrical ring r_lo < K <= r_hi, a_lo < Kpll <= a_hi
    // (Fill_array_cylindrical_ring); theta, Kpll about the axis dirn
    double a_lo, a_hi;
    int dirn;
    Cut cut;
};

// Columns go from memory to registers and back in transform order; a column
// without a mode to keep is not read.  One field at 256^3 FP64: 123 us with the
// tiles staged through LDS, now 76.  FILTER: flags & (8 | 16 | 32), cut.
template <typename T, int L, int CB, bool FILTER>
__global__ void __launch_bounds__(CB *(L / 8)) k_xinv_state(XinvArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= (FILTER ? x_tiles_cut<T>(g, CB, a.cut) : x_tiles(g, CB, false))) return;
    const ColTile<T, L, CB> t(g, FILTER ? x_tile_cut<T>(g, CB, a.cut, tile) : tile);
    const int j = t.j, ky = kwave(t.ly, g.ny), lz = t.lz;
    int zx0 = 1, zx1 = 0;
    if (a.flags & 1) dealias_rows(g, t.ly, lz, zx0, zx1);
    const bool slots = (a.flags & 2) != 0;
    bool need = t.live && (slots || zx0 > 0 || zx1 < L - 1);
    if (FILTER && kmag(g, 0, ky, lz) > a.r_hi) need = false;   // (K grows with |kx|)
    cpx<double> d[8];
    auto load = [&](int comp) {
        if (need) {
            col_load<false>(d, (const cpx<double> *)a.V[comp] + t.state0, t.steps, t.offs);
        } else {
#pragma unroll
            for (int s = 0; s < 8; s++) d[s] = mk<double>(0, 0);
        }
    };
    load(0);
    for (int i = threadIdx.x; i < L; i += CB * TPL) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    const X x{lds + t.c};
#pragma unroll 1
    for (int comp = 0; comp < a.ncomp; comp++) {
        cpx<T> v[8];
        const int jh = hidden(j);
        if (slots && t.live) {
#pragma unroll 1
            for (int s = 0; s < 8; s++) {
                const int kx = kwave(jh + TPL * s, g.nx);
                const int sl = band_slot(a.b, kx, ky, lz);
                if (sl >= 0 && in_band(g, a.b, kx, ky, lz))
                    ((cpx<double> *)a.slots)[sl * 3 + comp] =
                        ((const cpx<double> *)a.V[comp])[((size_t)(jh + TPL * s) * g.ny + t.ly) * g.nzc + lz];
            }
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            bool keep = !(lx >= zx0 && lx <= zx1);
            if constexpr (FILTER) {
                const int kx = kwave(lx, g.nx);
                const double K = kmag(g, kx, ky, lz);
                keep = keep && K > a.r_lo && K <= a.r_hi;
                if (a.flags & 48) {
                    // universal_ET.cc:909-911 (ring) and :929-931 (cylindrical ring)
                    const double q = (a.flags & 16) ? aniso_polar(g, kx, ky, lz, a.dirn) : aniso_kpll(g, kx, ky, lz, a.dirn);
                    keep = keep && ((q > a.a_lo && q <= a.a_hi) || (fabs(q) < kAnisEps && a.a_lo < kAnisEps));
                }
            }
            v[s] = keep ? cvt<T>(d[s]) : mk<T>(0, 0);
            settle(v[s]);
        }
        pin_memory_order();
        if (comp + 1 < a.ncomp) load(comp + 1);
        pin_memory_order();
        fft_exchange<L, +1>(v, x, tw, jh);
        pin_memory_order();
        if (t.inside) col_store<false>(v, (cpx<T> *)a.U[comp] + t.cw0, t.stepw, t.offt);
    }
}

// The strong reality condition on the kz = 0 and Nz/2 planes of the state (as
// k_reality) and the x-inverse of these columns, after the last stage of a
// step.  A column's mirrored rows are read where they are its own for
// lx > Nx/2 (and for lx = 0, ky < 0): no block writes a row that another reads.
// A block a component, both in one launch: 64^3 FP64 14 us a step, now 9; 512^3 160, now
// 123.
template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xinv_reality(XinvArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(g, CB, true)) return;
    const ColTile<T, L, CB> t(g, tile, true);
    const int j = t.j, ly = t.ly, lz = t.lz, ky = kwave(ly, g.ny);
    const bool nyquist = lz != 0;
    int zx0 = 1, zx1 = 0;
    if (a.flags & 1) dealias_rows(g, ly, lz, zx0, zx1);
    for (int i = threadIdx.x; i < L; i += CB * TPL) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    const X x{lds + t.c};
    const int comp = blockIdx.y;
    cpx<double> *V = (cpx<double> *)(comp == 0 ? a.V[0] : comp == 1 ? a.V[1] : a.V[2]);
    cpx<double> d[8];
    const int jh = hidden(j);
    auto mirrored = [&](int lx) { return (lx > g.nx / 2 && ky != g.ny / 2) || (lx == 0 && ky < 0); };
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int lx = jh + TPL * s;
        const bool m = mirrored(lx);
        const int rx = m && lx > 0 ? g.nx - lx : lx, ry = m && ly > 0 ? g.ny - ly : ly;
        const cpx<double> z = V[((size_t)rx * g.ny + ry) * g.nzc];
        d[s] = mk<double>(nyquist ? 0.0 : z.x, nyquist ? 0.0 : (m ? -z.y : z.y));
    }
    cpx<T> v[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int lx = jh + TPL * s;
        if (t.live && (nyquist || mirrored(lx))) V[((size_t)lx * g.ny + ly) * g.nzc + lz] = d[s];
        if ((a.flags & 2) && t.live) {
            const int kx = kwave(lx, g.nx), sl = band_slot(a.b, kx, ky, lz);
            if (sl >= 0 && in_band(g, a.b, kx, ky, lz)) ((cpx<double> *)a.slots)[sl * 3 + comp] = d[s];
        }
        v[s] = lx >= zx0 && lx <= zx1 ? mk<T>(0, 0) : cvt<T>(d[s]);
        settle(v[s]);
    }
    fft_exchange<L, +1>(v, x, tw, jh);
    pin_memory_order();
    if (t.inside) col_store<false>(v, (cpx<T> *)(comp == 0 ? a.U[0] : comp == 1 ? a.U[1] : a.U[2]), t.stepw, t.offt);
}

// ---------------------------------------------------------------------------
// x-forward of T work fields into FP64 spectral outputs (last pass of the 3D
// forward transform), scaled.
// ---------------------------------------------------------------------------
struct XfwdArgs {
    void *W[3];
    double *out[3];
    const void *tw;
    Grid g;
    double scale;
    int ncomp;
};

template <typename T, int L, int CB>
__global__ void __launch_bounds__(CB *(L / 8)) k_xfwd_spec(XfwdArgs a)
{
    constexpr int TPL = L / 8;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    __shared__ cpx<T> tw[L];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= x_tiles(a.g, CB, false)) return;
    const ColTile<T, L, CB> t(a.g, tile);
    cpx<T> v[8];
    col_load<false>(v, (const cpx<T> *)a.W[0] + t.cw0, t.stepw, t.offt);
    for (int i = threadIdx.x; i < L; i += CB * TPL) tw[i] = ((const cpx<T> *)a.tw)[i];
    lds_barrier();
    const X x{lds + t.c};
#pragma unroll 1
    for (int comp = 0; comp < a.ncomp; comp++) {
        fft_exchange<L, -1>(v, x, tw, hidden(t.j));
        cpx<double> o[8];
#pragma unroll
        for (int s = 0; s < 8; s++) o[s] = a.scale * cvt<double>(v[s]);
        pin_memory_order();
        if (comp + 1 < a.ncomp) col_load<false>(v, (const cpx<T> *)a.W[comp + 1] + t.cw0, t.stepw, t.offt);
        pin_memory_order();
        if (t.live) col_store<false>(o, (cpx<double> *)a.out[comp] + t.state0, t.steps, t.offs);
    }
}

template <typename T, int M, int W>
__global__ void __launch_bounds__(64 * W) k_z_c2r(ZArgs a)
{
    constexpr int TPL = M / 8;
    constexpr int LP = lpad_len(M);
    __shared__ cpx<T> lds[ZLines<M, W>::LPB * LP], ldw[2 * M];
    const ZTwiddles<T, M> tw(ldw, a.twm, a.twn);
    const ZLines<M, W> z(a.g);
    if (z.spare) return;
    const int li = z.li, j = z.j;
    const size_t line = z.line, lsafe = z.safe;
    for (int comp = 0; comp < a.ncomp; comp++) {
        const cpx<T> *X = (const cpx<T> *)a.in[comp] + lsafe * a.g.nzp;
        cpx<T> v[8];
        zline_c2r<T, M>(v, X, lds + li * LP, tw, j);
        if (z.valid) {
            double *R = (double *)a.out[comp] + line * (size_t)(2 * M + 2);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int n = j + TPL * s;
                ((cpx<double> *)R)[n] = cvt<double>(v[s]);
            }
            if (j == 0) ((cpx<double> *)R)[M] = mk<double>(0, 0);
        }
        line_sync();
    }
}

template <typename T, int M, int W>
__global__ void __launch_bounds__(64 * W) k_z_r2c(ZArgs a)
{
    constexpr int TPL = M / 8;
    constexpr int LP = lpad_len(M);
    __shared__ cpx<T> lds[ZLines<M, W>::LPB * LP], ldw[2 * M];
    const ZTwiddles<T, M> tw(ldw, a.twm, a.twn);
    const ZLines<M, W> z(a.g);
    if (z.spare) return;
    const int li = z.li, j = z.j;
    const size_t line = z.line, lsafe = z.safe;
    for (int comp = 0; comp < a.ncomp; comp++) {
        const cpx<double> *R = (const cpx<double> *)((const double *)a.in[comp] + lsafe * (size_t)(2 * M + 2));
        cpx<T> v[8];
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = cvt<T>(R[j + TPL * s]);
        cpx<T> *X = (cpx<T> *)a.out[comp] + lsafe * a.g.nzp;
        zline_r2c_post<T, M>(v, X, lds + li * LP, tw, j, z.valid, a.g.nzp - M);
    }
}

// z pass of the nonlinear term.  NS: products u_a u_b for the pairs
// (0,0),(1,1),(2,2),(0,1),(1,2),(2,0) -- the six real-space products of
// Compute_nlin_diag / Compute_nlin_offdiag (compute_diag_offdiag.cc:47-112);
// a.ncomp == 5: the trace-shifted five u_x^2 - u_z^2, u_y^2 - u_z^2, u_x u_y,
// u_y u_z, u_z u_x (the nonlinear term less the gradient i K F[u_z^2], which
// the pressure projection removes).
// Giver: out[3*i + j] = u_j w_i (compute_diag_offdiag.cc:329-414).
// Bound by HBM.  The twiddles sit in LDS: read from global memory, those of
// each product waited for the stores of the one before (loads and stores
// retire in order) and took 168 of the 264 memory instructions of a wave.
// Rows are written whole, and non-temporally where the fields pass the
// memory-side cache.  512^3, per launch: FP64 2125 -> 1736 us (5.0 TB/s), FP32
// 1363 -> 830 us (5.2 TB/s).
// FP32 lines of 256 points (512-point z axis): four waves per SIMD (the
// allocation fits 128 VGPRs without spills).
// FIVE: the NS form with the five trace-shifted products (an instance of its
// own: with both NS forms in one kernel the FP32 instance spilled under its
// four-wave bound); with GIVER, the eight trace-shifted products of the MHD
// stage: P_xx - P_zz, P_yy - P_zz and the six off-diagonal ones (P_zz is
// not stored).
template <typename T, int M, bool GIVER, bool FIVE, bool NT, int W>
__global__ void __launch_bounds__(64 * W, (sizeof(T) == 4 && !GIVER && M == 256) ? 4 : 1) k_z_products(ZArgs a)
{
    constexpr int TPL = M / 8;
    constexpr int LPB = ZLines<M, W>::LPB;
    constexpr int LP = lpad_len(M);
    __shared__ cpx<T> lds[LPB * LP], ldw[2 * M];
    const ZLines<M, W> z(a.g);
    const int li = z.li, j = z.j;
    const size_t line = z.line, lsafe = z.safe;
    const bool valid = z.valid;
    cpx<T> *L = lds + li * LP;
    // the three input lines are loaded before the first transform: their
    // loads are in flight together
    constexpr bool LIM = GIVER && !FIVE;
    cpx<T> u[3][8], xm[3];
#pragma unroll
    for (int c = 0; c < 3; c++)
        zline_load<T, M, NT, LIM>(u[c], xm[c], (const cpx<T> *)a.in[c] + lsafe * a.g.nzp, j, a.lim_u);
    const ZTwiddles<T, M> tw(ldw, a.twm, a.twn);
    if (z.spare) return;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        zline_c2r_from<T, M>(u[c], xm[c], L, tw, j);
        line_sync();
    }
    if (!GIVER && a.tape[0] && valid) {
        // the adjoint's record of u = I(D V) for this stage
#pragma unroll
        for (int c = 0; c < 3; c++) {
            cpx<T> *tp = (cpx<T> *)a.tape[c] + line * M;
#pragma unroll
            for (int s = 0; s < 8; s++) tp[j + TPL * s] = u[c][s];
        }
    }
    auto emit = [&](cpx<T> *p, int o) {
        cpx<T> *X = (cpx<T> *)a.out[o] + lsafe * a.g.nzp;
        zline_r2c_post<T, M, NT, LIM>(p, X, L, tw, j, valid, a.g.nzp - M, a.lim_out);
    };
    if constexpr (!GIVER && FIVE) {
        // the cross products first, then the two shifted squares (u_z is
        // last used there)
        const int pa[3] = {0, 1, 2};
        const int pb[3] = {1, 2, 0};
#pragma unroll
        for (int o = 0; o < 3; o++) {
            cpx<T> p[8];
#pragma unroll
            for (int s = 0; s < 8; s++) p[s] = mk<T>(u[pa[o]][s].x * u[pb[o]][s].x, u[pa[o]][s].y * u[pb[o]][s].y);
            emit(p, 2 + o);
        }
#pragma unroll
        for (int o = 0; o < 2; o++) {
            cpx<T> p[8];
#pragma unroll
            for (int s = 0; s < 8; s++)
                p[s] = mk<T>(u[o][s].x * u[o][s].x - u[2][s].x * u[2][s].x,
                             u[o][s].y * u[o][s].y - u[2][s].y * u[2][s].y);
            emit(p, o);
        }
    } else if constexpr (!GIVER) {
        const int pa[6] = {0, 1, 2, 0, 1, 2};
        const int pb[6] = {0, 1, 2, 1, 2, 0};
#pragma unroll
        for (int o = 0; o < 6; o++) {
            cpx<T> p[8];
#pragma unroll
            for (int s = 0; s < 8; s++) p[s] = mk<T>(u[pa[o]][s].x * u[pb[o]][s].x, u[pa[o]][s].y * u[pb[o]][s].y);
            emit(p, o);
        }
    } else if constexpr (FIVE) {
        // w_z first: P_zz = u_z w_z is kept, in this thread's own LDS slots
        // (registers would cost the FP64 instance half its occupancy), for the
        // two shifted diagonal products
        __shared__ cpx<T> dl[LPB * M];
        cpx<T> *D = dl + li * M;
#pragma unroll 1
        for (int ii = 0; ii < 3; ii++) {
            const int i = ii == 0 ? 2 : ii - 1;
            cpx<T> w[8];
            zline_c2r<T, M, NT>(w, (const cpx<T> *)a.in[3 + i] + lsafe * a.g.nzp, L, tw, j);
            line_sync();
            if (ii == 0) {
#pragma unroll
                for (int s = 0; s < 8; s++) D[j + TPL * s] = mk<T>(u[2][s].x * w[s].x, u[2][s].y * w[s].y);
            }
#pragma unroll
            for (int jj = 0; jj < 3; jj++) {
                if (jj == i && i == 2) continue;
                cpx<T> p[8];
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    p[s] = mk<T>(u[jj][s].x * w[s].x, u[jj][s].y * w[s].y);
                    if (jj == i) p[s] = p[s] - D[j + TPL * s];
                }
                emit(p, 3 * i + jj);
            }
        }
    } else {
#pragma unroll 1
        for (int i = 0; i < 3; i++) {
            cpx<T> w[8];
            zline_c2r<T, M, NT, LIM>(w, (const cpx<T> *)a.in[3 + i] + lsafe * a.g.nzp, L, tw, j, a.lim_w);
            line_sync();
#pragma unroll
            for (int jj = 0; jj < 3; jj++) {
                cpx<T> p[8];
#pragma unroll
                for (int s = 0; s < 8; s++) p[s] = mk<T>(u[jj][s].x * w[s].x, u[jj][s].y * w[s].y);
                emit(p, 3 * i + jj);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Fused x pass of the nonlinear term and the Lawson RK4 stage.
// ---------------------------------------------------------------------------
struct XnlArgs {
    void *P[9];
    double *V[3];
    double *acc[3];  // stage accumulator, FP64 (padded work layout)
    void *U[3];
    double *out[3];
    const double *slots_in;
    double *slots_out;
    const void *tw;
    Grid g;
    Band b;
    RkParams rk;
    Cut cut;   // giver form
};

// alpha = eps / (2 E_band) with E_band = sum w |V|^2 over the band modes,
// w = 1/2 on kz = 0 (Get_local_energy weights, FFF_pencil_energy.cc:59-67),
// summed by the NT threads of the block in a fixed order (red: 16 values of
// LDS; every thread of the block calls it).
template <int NT>
__device__ __forceinline__ double band_alpha(const Grid &g, const Band &b, const double *slots, double *red)
{
    const int n = band_nslots(b);
    double e = 0.0;
    for (int s = threadIdx.x; s < n; s += NT) {
        const int kz = s % (b.h[2] + 1);
        const int ky = (s / (b.h[2] + 1)) % (2 * b.h[1] + 1) - b.h[1];
        const int kx = s / ((b.h[2] + 1) * (2 * b.h[1] + 1)) - b.h[0];
        const double K = kmag(g, kx, ky, kz);
        if (K > b.r_in && K <= b.r_out) {
            const double w = kz == 0 ? 0.5 : 1.0;
            for (int c = 0; c < 3; c++) {
                const double re = slots[2 * (s * 3 + c)], im = slots[2 * (s * 3 + c) + 1];
                e += w * (re * re + im * im);
            }
        }
    }
    // lanes past the block's last thread hold nothing to add
    constexpr int NW = (NT + 63) / 64;
    for (int off = 32; off > 0; off >>= 1) {
        const double t = __shfl_down(e, off, 64);
        if ((int)(threadIdx.x & 63) + off < 64 && (int)threadIdx.x + off < NT) e += t;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = e;
    lds_barrier();
    double t = 0.0;
    for (int w = 0; w < NW; w++) t += red[w];
    return t > 0.0 ? b.eps / (2.0 * t) : 0.0;
}

// Where the force of the modes of a column lies in b.force, in modes: row kx at
// place + kx step.
__device__ __forceinline__ void force_place(const Grid &g, const Band &b, int ky, int ly, int lz, int &place, int &step)
{
    step = b.kind == 1 ? (2 * b.h[1] + 1) * (b.h[2] + 1) : g.ny * g.nzp;
    place = b.kind == 1 ? band_slot(b, 0, ky, lz) : (g.nx / 2 - 1) * step + ly * g.nzp + lz;
}

// Random band forcing of one mode (kind 2; compute_force_random.cc:65-130,
// force_amp_phase.cc:119-170, FFF_pencil_inline.h:234-248): helical
// amplitudes sqrt((e_k +- h_k/K) / tau) with phases 2 pi U(seed, 2m),
// 2 pi U(seed, 2m + 1), m = (lx Ny + ly)(Nz/2+1) + lz; U1 = i (F- - F+),
// U2 = F- + F+ in the Craya basis; Cartesian components about z.
__device__ void random_force_mode(const Grid &g, const Band &b, int lx, int ly, int lz, int kx, int ky, double K,
                                  cpx<double> *F)
{
    const int i = (int)ceil(K);
    const double e = b.shell_eh[2 * i], h = b.shell_eh[2 * i + 1];
    const double ap = sqrt((e + h / K) / b.tau), am = sqrt((e - h / K) / b.tau);
    const uint64_t m = ((uint64_t)lx * g.ny + ly) * g.nzc + lz;
    const double twopi = 6.28318530717958647692;
    const double php = twopi * uniform01(b.seed, 2 * m), phm = twopi * uniform01(b.seed, 2 * m + 1);
    const cpx<double> Fp = mk<double>(ap * cos(php), ap * sin(php)), Fm = mk<double>(am * cos(phm), am * sin(phm));
    const cpx<double> d = Fm - Fp;
    const cpx<double> U1 = mk<double>(-d.y, d.x), U2 = Fm + Fp;
    const double th = aniso_polar(g, kx, ky, lz, 3), ph = aniso_azimuth(g, kx, ky, lz, 3);
    const double st = sin(th), ct = cos(th), sp = sin(ph), cp = cos(ph);
    F[0] = sp * U1 + (ct * cp) * U2;
    F[1] = (-cp) * U1 + (sp * ct) * U2;
    F[2] = (-st) * U2;
}

#if TG_LEN_UNIT == 0
// The random force of the band's modes (r_in < K <= r_out).  The phases hold for a
// whole call, so they are drawn once here: within the x pass their sines and
// cosines were most of its instructions (0.5 ms of a 512^3 FP64 step).
__global__ void k_random_force(Grid g, Band b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= band_nslots(b)) return;
    const int kz = i % (b.h[2] + 1);
    const int ky = (i / (b.h[2] + 1)) % (2 * b.h[1] + 1) - b.h[1];
    const int kx = i / ((b.h[2] + 1) * (2 * b.h[1] + 1)) - b.h[0];
    // the indices of the mode; k = -N/2 is not one
    const int lx = kx >= 0 ? kx : kx + g.nx, ly = ky >= 0 ? ky : ky + g.ny;
    if (kwave(lx, g.nx) != kx || kwave(ly, g.ny) != ky || kz >= g.nzc || !in_band(g, b, kx, ky, kz)) return;
    cpx<double> F[3];
    random_force_mode(g, b, lx, ly, kz, kx, ky, kmag(g, kx, ky, kz), F);
    int place, step;
    force_place(g, b, ky, ly, kz, place, step);
#pragma unroll
    for (int c = 0; c < 3; c++) ((cpx<double> *)b.force)[(size_t)3 * (place + kx * step) + c] = F[c];
}

hipError_t launch_random_force(const Grid &g, const Band &b, hipStream_t st)
{
    const int n = band_nslots(b);
    hipLaunchKernelGGL(k_random_force, dim3((n + 63) / 64), dim3(64), 0, st, g, b);
    return hipGetLastError();
}
#endif

// The x pass's products, in the reference's accumulation order
// (compute_diag_offdiag.cc:47-112 for NS, :329-414 for the giver form).
enum {
    XNL_SIX = 0,    // NS products xx, yy, zz, xy, yz, zx
    XNL_GIVER = 1,  // P[3i+j] = FT[u_j w_i]: i K_j P to N_i
    XNL_TRANS = 2,  // transposed (MHD: N-_j = sum_i d_i(Z+_i Z-_j)): i K_i P to N_j
    XNL_FIVE = 3,   // trace-shifted xx - zz, yy - zz, xy, yz, zx, where the nonlinear
                    // term is only used projected (its gradient part i K F[u_z^2]
                    // drops out)
};
constexpr int xnl_products(int mode) { return mode == XNL_SIX ? 6 : (mode == XNL_FIVE ? 5 : 9); }
constexpr int xnl_index(int mode, int pi)
{
    constexpr int giver[9] = {0, 4, 8, 3, 1, 7, 5, 2, 6};
    return mode == XNL_SIX || mode == XNL_FIVE ? pi : giver[pi];
}
// product index p of mode: the axis d whose i K_d FT[p] is added to N_i, -1: none
constexpr int xnl_axis(int mode, int p, int i)
{
    if (mode == XNL_GIVER) return p / 3 == i ? p % 3 : -1;
    if (mode == XNL_TRANS) return p % 3 == i ? p / 3 : -1;
    constexpr int sel[6][3] = {{0, -1, -1}, {-1, 1, -1}, {-1, -1, 2}, {1, 0, -1}, {-1, 2, 1}, {2, -1, 0}};
    return sel[mode == XNL_FIVE && p >= 2 ? p + 1 : p][i];
}

// Bound by HBM and by the one block of two waves a SIMD that its registers
// leave: the next tile is always in flight.  Columns go from memory to
// registers in the transform's own order (ColX) and back; LDS holds the
// exchanges, the twiddles and the viscous factors.  Every value is settled
// where it is formed, and each stage is an instance of its own: with the four
// stages, the hyperviscosity loops and the random phases inlined per point the
// kernel was 300 KB of instructions, mostly fetched from L2 (and the stages'
// registers, allocated together, spilled).  512^3, per launch, mean of the four
// stages: FP64 5170 -> 3620 us (4.8 TB/s), FP32 4550 -> 3150 us; 64^3 FP64 54 ->
// 19 us, 240x160x96 348 -> 137 us; a step of 1024 x 256 x 512 (64-byte rows, one
// block a CU) FP64 58.5 -> 38.2 ms, FP32 42.5 -> 27.2 ms.
template <typename T, int L, int CB, int MODE, int ST, bool NT>
__global__ void __launch_bounds__(CB *(L / 8), 2) k_x_nlin(XnlArgs a)
{
    constexpr int TPL = L / 8;
    // non-temporal access of whole 128-byte lines only (the unpadded state rows
    // share their lines with the neighbouring tiles)
    constexpr bool NTW = NT && CB * sizeof(cpx<T>) >= 128, NTA = NT && CB * sizeof(cpx<double>) >= 128;
    using X = ColX<T, L, CB>;
    __shared__ cpx<T> lds[X::SIZE];
    // twiddles are read from LDS: a load from global memory between the FFT
    // passes would wait for the next tile's loads in flight
    __shared__ cpx<T> tw[L];
    __shared__ double red[16];
    // the viscous factors of this thread's points (their registers would
    // spill): exp(-nu K^2 dt/2), stage 4 exp(-nu K^2 dt), stage 1 both
    __shared__ double visc[ST == 1 ? 2 : 1][ST ? 8 * CB * TPL : 1];
    const Grid &g = a.g;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    constexpr bool CUT = MODE == XNL_GIVER;
    if (tile >= (CUT ? x_tiles_cut<T>(g, CB, a.cut) : x_tiles(g, CB, false))) return;
    const ColTile<T, L, CB> t(g, CUT ? x_tile_cut<T>(g, CB, a.cut, tile) : tile);
    const int j = t.j, ly = t.ly, lz = t.lz, cw0 = t.cw0;
    const bool live = t.live;
    const size_t stepw = t.stepw, steps = t.steps, state0 = t.state0;
    const uint32_t offt = t.offt, offw = t.offw, offs = t.offs;
    const int ky = kwave(ly, g.ny);
    const double Ky = ky * g.kf[1], Kz = lz * g.kf[2];
    const T sc = (T)a.rk.scale;
    const T Kyt = (T)Ky, Kzt = (T)Kz;
    constexpr bool NS = MODE == XNL_SIX || MODE == XNL_FIVE;
    constexpr int NP = xnl_products(MODE);
    const bool want_rhs = NS && (ST > 0 || a.rk.write_rhs);

    cpx<T> cur[8];
    col_load<NTW>(cur, (const cpx<T> *)a.P[0] + cw0, stepw, offt);
    for (int i = threadIdx.x; i < L; i += CB * TPL) tw[i] = ((const cpx<T> *)a.tw)[i];
    // whether a column of this tile can hold forced modes; the alpha forcing's
    // coefficient is summed by the block (one thread summing all the slots
    // took 70 us of a 128^3 stage)
    const bool band_tile = NS && a.b.kind != 0 && (t.WIDE || (abs(ky) <= a.b.h[1] && t.lz0 <= a.b.h[2]));
    double alpha = 0.0;
    if (band_tile && a.b.kind == 1 && want_rhs) alpha = band_alpha<CB * TPL>(g, a.b, a.slots_in, red);
    unsigned forced = 0;   // bit s: row j + TPL s of this column is forced
    if (band_tile && live)
        for (int s = 0; s < 8; s++) {
            const int kx = kwave(j + TPL * s, g.nx);
            if (band_slot(a.b, kx, ky, lz) >= 0 && in_band(g, a.b, kx, ky, lz)) forced |= 1u << s;
        }
    lds_barrier();
    const X x{lds + t.c};

    // --- forward x-FFT of the products and the divergence-form sum ---
    // Unrolled over the products: each adds to the one or two components its
    // derivatives belong to, and the next one (at the end the state of the
    // first component) is in flight while it is transformed.
    cpx<T> N[3][8];
#pragma unroll
    for (int s = 0; s < 8; s++) N[0][s] = N[1][s] = N[2][s] = mk<T>(0, 0);
    cpx<double> v0[8];
    auto product = [&](auto pc, cpx<T> *v, cpx<T> *next) {
        constexpr int PI = decltype(pc)::value;
        pin_memory_order();
        if constexpr (PI + 1 < NP) col_load<NTW>(next, (const cpx<T> *)a.P[xnl_index(MODE, PI + 1)] + cw0, stepw, offt);
        else if (ST > 0) col_load<false>(v0, (const cpx<double> *)a.V[0] + state0, steps, offs);
        pin_memory_order();
        const int jh = hidden(j);
        fft_exchange<L, -1>(v, x, tw, jh);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const T Kx = (T)(kwave(jh + TPL * s, g.nx) * g.kf[0]);
            const cpx<T> q = sc * v[s];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                constexpr int P = xnl_index(MODE, PI);
                const int d = xnl_axis(MODE, P, i);
                if (d >= 0) {
                    N[i][s] = N[i][s] + mul_i(d == 0 ? Kx : (d == 1 ? Kyt : Kzt), q);
                    settle(N[i][s]);
                }
            }
        }
    };
    cpx<T> alt[8];
    auto pair = [&](auto pc) {
        constexpr int PI = decltype(pc)::value;
        if constexpr (PI < NP) product(std::integral_constant<int, PI>{}, cur, alt);
        if constexpr (PI + 1 < NP) product(std::integral_constant<int, PI + 1>{}, alt, cur);
    };
    pair(std::integral_constant<int, 0>{});
    pair(std::integral_constant<int, 2>{});
    pair(std::integral_constant<int, 4>{});
    pair(std::integral_constant<int, 6>{});
    pair(std::integral_constant<int, 8>{});

    // --- force, pressure projection, negation (Compute_force_TO_rhs), in
    // place on N: N <- -(N - F + i K p), p = i K.(N - F) / K^2 (computed in
    // FP64, stored in the transform precision); the forced modes in a second
    // turn, so that all others take one code in every tile ---
    auto project = [&](auto fc) {
        constexpr bool FORCED = decltype(fc)::value;
        const int jh = hidden(j);
        int place = 0, step = 0;
        if constexpr (FORCED) force_place(g, a.b, ky, ly, lz, place, step);
        const double fscale = a.b.kind == 1 ? alpha : 1.0;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int lx = jh + TPL * s;
            const int kx = kwave(lx, g.nx);
            const double Kx = kx * g.kf[0];
            const bool f_mode = (forced & (1u << s)) != 0;
            if (FORCED && !f_mode) continue;
            cpx<double> n0 = cvt<double>(N[0][s]), n1 = cvt<double>(N[1][s]), n2 = cvt<double>(N[2][s]);
            if constexpr (FORCED) {
                // the stage input's band modes, or the random force itself
                const cpx<double> *sv = (const cpx<double> *)a.b.force + (size_t)3 * (uint32_t)(place + kx * step);
                n0 = n0 - fscale * sv[0];
                n1 = n1 - fscale * sv[1];
                n2 = n2 - fscale * sv[2];
            }
            cpx<double> div = mul_i(Kx, n0);
            div = div + mul_i(Ky, n1);
            div = div + mul_i(Kz, n2);
            const double kxs = Kx * Kx;
            const double ks = (kxs + Ky * Ky) + Kz * Kz;
            cpx<double> pr = mk<double>(0, 0);
            if (!(lx == 0 && ly == 0 && lz == 0)) pr = mk<double>(div.x / ks, div.y / ks);
            n0 = n0 + mul_i(Kx, pr);
            n1 = n1 + mul_i(Ky, pr);
            n2 = n2 + mul_i(Kz, pr);
            const cpx<T> r0 = cvt<T>(mk<double>(-n0.x, -n0.y)), r1 = cvt<T>(mk<double>(-n1.x, -n1.y)),
                         r2 = cvt<T>(mk<double>(-n2.x, -n2.y));
            const bool keep = !FORCED && f_mode;
            N[0][s] = mk<T>(keep ? N[0][s].x : r0.x, keep ? N[0][s].y : r0.y);
            N[1][s] = mk<T>(keep ? N[1][s].x : r1.x, keep ? N[1][s].y : r1.y);
            N[2][s] = mk<T>(keep ? N[2][s].x : r2.x, keep ? N[2][s].y : r2.y);
#pragma unroll
            for (int i = 0; i < 3; i++) settle(N[i][s]);
            if (s % 2) __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (want_rhs) {
        project(std::false_type{});
        if (band_tile) project(std::true_type{});
    }

    if constexpr (ST == 0) {
        // Compute_nlin (and optionally Compute_rhs) output, FP64 boundary layout
        if (live) {
#pragma unroll
            for (int comp = 0; comp < 3; comp++) {
                cpx<double> o[8];
#pragma unroll
                for (int s = 0; s < 8; s++) o[s] = cvt<double>(N[comp][s]);
                col_store<false>(o, (cpx<double> *)a.out[comp] + state0, steps, offs);
            }
        }
        return;
    }

    // --- Lawson RK4 stage algebra (RK.cc:91-170, Tadvance_functions.cc:298-324,566-570) ---
    // V: FP64 state, boundary layout; acc: FP64, padded work layout (the RK
    // state accumulation stays FP64 whatever the transform precision).  The
    // next component's state is loaded before this one's results are stored
    // (loads and stores retire in order, so that the wait for it does not
    // wait for those stores).
    const double dt = a.rk.dt;
    const double c_half = 0.5 * dt, c_one = 1.0 * dt;
    const double c_sixth = (1.0 / 6) * dt, c_third = (1.0 / 3) * dt;
    int zx0, zx1;   // rows of this column that the dealias mask zeroes (a pad column: all)
    dealias_rows(g, ly, lz, zx0, zx1);
    if (!live) { zx0 = 0; zx1 = L - 1; }
    if constexpr (ST > 0) {
        {
            const int jh = hidden(j);
#pragma unroll 2
            for (int s = 0; s < 8; s++) {
                const double Kx = kwave(jh + TPL * s, g.nx) * g.kf[0];
                const double kxs = Kx * Kx;
                const double ks = (kxs + Ky * Ky) + Kz * Kz;
                const double kp = hyper_power(a.rk.hq, ks);
                if (ST < 4) visc[0][s * CB * TPL + threadIdx.x] = exp((a.rk.fh + a.rk.fhh * kp) * ks);
                if (ST == 1 || ST == 4)
                    visc[ST == 1][s * CB * TPL + threadIdx.x] = exp((a.rk.f1 + a.rk.f1h * kp) * ks);
            }
        }
        // (each thread reads its own entries only)
        auto Eh = [&](int s) { return visc[0][s * CB * TPL + threadIdx.x]; };
        auto E1 = [&](int s) { return visc[ST == 1][s * CB * TPL + threadIdx.x]; };
        cpx<double> ac[8];
        if (ST >= 2) col_load<NTA>(ac, (const cpx<double> *)a.acc[0] + cw0, stepw, offw);
        double chk = 0.0;   // stage 4: NaN after a non-finite value
        // SLOTS: the undealiased stage input of forced modes goes to the slots
        auto algebra = [&](auto kc, auto slc, cpx<T> *v) {
            constexpr int K = decltype(kc)::value;
            constexpr bool SLOTS = decltype(slc)::value;
            const int jh = hidden(j);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int lx = jh + TPL * s;
                const cpx<double> r = cvt<double>(N[K][s]);
                cpx<double> vn;
                if constexpr (ST == 1) {
                    cpx<double> d0 = v0[s];
                    if (lx >= zx0 && lx <= zx1) d0 = mk<double>(0, 0);
                    ac[s] = c_sixth * (E1(s) * r);
                    vn = Eh(s) * (d0 + c_half * r);
                } else if constexpr (ST == 2) {
                    ac[s] = ac[s] + c_third * (Eh(s) * r);
                    vn = Eh(s) * v0[s] + c_half * r;
                } else if constexpr (ST == 3) {
                    ac[s] = ac[s] + c_third * (Eh(s) * r);
                    vn = Eh(s) * (Eh(s) * v0[s] + c_one * r);
                } else {
                    ac[s] = ac[s] + c_sixth * r;
                    vn = E1(s) * v0[s] + ac[s];
                    ac[s] = vn;   // the new state
                    chk += 0.0 * vn.x + 0.0 * vn.y;
                }
                if (SLOTS && (forced & (1u << s)))
                    ((cpx<double> *)a.slots_out)[band_slot(a.b, kwave(lx, g.nx), ky, lz) * 3 + K] = vn;
                if (lx >= zx0 && lx <= zx1) vn = mk<double>(0, 0);
                v[s] = cvt<T>(vn);
            }
        };
        auto rk_comp = [&](auto kc) {
            constexpr int K = decltype(kc)::value;
            cpx<T> v[8];
            if (band_tile && a.b.kind == 1) algebra(kc, std::true_type{}, v);
            else algebra(kc, std::false_type{}, v);
            pin_memory_order();
            if constexpr (K < 2) col_load<false>(v0, (const cpx<double> *)a.V[K + 1] + state0, steps, offs);
            if (ST == 4) {
                if (live) col_store<false>(ac, (cpx<double> *)a.V[K] + state0, steps, offs);
            } else {
                if (t.inside) col_store<NTA>(ac, (cpx<double> *)a.acc[K] + cw0, stepw, offw);
            }
            if (ST >= 2 && K < 2)
                col_load<NTA>(ac, (const cpx<double> *)a.acc[K < 2 ? K + 1 : 2] + cw0, stepw, offw);
            pin_memory_order();
            fft_exchange<L, +1>(v, x, tw, hidden(j));
            pin_memory_order();
            if (t.inside) col_store<NTW>(v, (cpx<T> *)a.U[K] + cw0, stepw, offt);
        };
        rk_comp(std::integral_constant<int, 0>{});
        rk_comp(std::integral_constant<int, 1>{});
        rk_comp(std::integral_constant<int, 2>{});
        if (ST == 4 && chk != 0.0 && live && a.rk.nonfinite) *a.rk.nonfinite = 1;
    }
}

#if TG_LEN_UNIT == 0
// ---------------------------------------------------------------------------
// Strong reality condition (FFF_pencil_basic.cc:139-179) and dealias.
// ---------------------------------------------------------------------------
struct PlaneArgs {
    double *V[3];
    Grid g;
    int ncomp;
};

__global__ void k_reality(PlaneArgs a)
{
    const Grid &g = a.g;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= g.nx * g.ny) return;
    const int lx = idx / g.ny, ly = idx % g.ny;
    const int ky = kwave(ly, g.ny);
    for (int comp = 0; comp < a.ncomp; comp++) {
        cpx<double> *A = (cpx<double> *)a.V[comp];
        const size_t t = ((size_t)lx * g.ny + ly) * g.nzc;
        int src = -1;
        if (lx > g.nx / 2 && ky != g.ny / 2) {
            const int mkx = -kwave(lx, g.nx);
            const int mky = -ky;
            const int iy = mky >= 0 ? mky : mky + g.ny;
            src = mkx * g.ny + iy;
        } else if (lx == 0 && ky < 0) {
            src = -ky;
        }
        if (src >= 0) A[t] = conj(A[(size_t)src * g.nzc]);
        A[t + g.nzc - 1] = mk<double>(0, 0);
    }
}

__global__ void k_dealias(PlaneArgs a)
{
    const Grid &g = a.g;
    const size_t n = (size_t)g.nx * g.ny * g.nzc;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int lz = i % g.nzc;
        const int ly = (i / g.nzc) % g.ny;
        const int lx = i / ((size_t)g.nzc * g.ny);
        if (dealias_zero(g, lx, ly, lz))
            for (int comp = 0; comp < a.ncomp; comp++) ((cpx<double> *)a.V[comp])[i] = mk<double>(0, 0);
    }
}

#endif  // TG_LEN_UNIT == 0

// ---------------------------------------------------------------------------
// Per-length launch functions (instantiated in the length units) and the
// launchers with their size dispatch.
// ---------------------------------------------------------------------------
template <typename T, int LL>
hipError_t colfft_len(const ColArgs &a, int dir, int nfields, hipStream_t st)
{
    // Tiles of 128-byte rows (8 FP64 or 16 FP32 columns), fewer only where a
    // block would pass 1024 threads: with rows of 64 bytes the in-place pass of
    // five 512^3 FP64 fields takes 2461 us against 2017, and at 1024 points,
    // where the wide tile leaves one block per CU, 2485 against 2152.
    constexpr int CB = colx_block<T>(LL, 1024);
    // Non-temporal loads and stores where the pass streams more than the 256
    // MiB memory-side cache holds (five 512^3 FP64 fields 2017 -> 1892 us in a
    // loop of the pass alone, 445 -> 381 us per field within the step); 128^3
    // FP32 lost 5% in the z pass that follows.  Not where a CU holds one block
    // (1024 points FP64 2152 against 2226 us) or the rows are half lines.
    constexpr bool STREAM = LL >= kStreamLength && CB * sizeof(cpx<T>) >= 128 &&
                            2 * ColX<T, LL, CB>::SIZE * sizeof(cpx<T>) <= 160 * 1024;
    dim3 grid(x_grid(a.nouter * ((a.ncol + CB - 1) / CB)), nfields);
    const dim3 block(CB * (LL / 8));
    const bool nt = STREAM && stream_bytes((size_t)nfields * a.nouter * a.outer_stride * sizeof(cpx<T>));
    const bool cut = a.keep < LL / 2;
    auto go = [&](auto dc, auto ntc) {
        constexpr int DIR = decltype(dc)::value;
        constexpr bool NT = decltype(ntc)::value;
        if (cut) hipLaunchKernelGGL((k_colfft<T, LL, DIR, CB, NT, true>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k_colfft<T, LL, DIR, CB, NT, false>), grid, block, 0, st, a);
    };
    using fwd = std::integral_constant<int, -1>;
    using inv = std::integral_constant<int, +1>;
    using stream = std::bool_constant<STREAM>;
    if (dir < 0 && nt) go(fwd{}, stream{});
    else if (dir < 0) go(fwd{}, std::false_type{});
    else if (nt) go(inv{}, stream{});
    else go(inv{}, std::false_type{});
    return hipGetLastError();
}

// Columns of the plain x passes' tiles: 16, whose 256 bytes of an unpadded state
// row lie in three 128-byte lines (8 columns in two, half of each another
// tile's), while a block has at most 1024 threads.  256^3 FP64, 8 columns: inverse
// 85 us, forward 60; 16: 76 and 53; 512 x 256 x 256: 161 and 151 us, 148 and 128.
// (The filtered inverse needs more registers than such a block has.)
__host__ __device__ constexpr int plain_block(int L)
{
    int cb = 16;
    while (cb * (L / 8) < 64) cb *= 2;
    while (cb * (L / 8) > 1024) cb /= 2;
    return cb;
}

template <typename T, int LL>
hipError_t xinv_state_len(const XinvArgs &a, hipStream_t st)
{
    constexpr int CB = colx_block<T>(LL, 512), PB = plain_block(LL);
    const dim3 grid(x_grid(x_tiles(a.g, CB, (a.flags & 4) != 0))), block(CB * (LL / 8));
    if (a.flags & 4) hipLaunchKernelGGL((k_xinv_reality<T, LL, CB>), dim3(grid.x, a.ncomp), block, 0, st, a);
    else if (a.flags & 56)
        hipLaunchKernelGGL((k_xinv_state<T, LL, CB, true>), dim3(x_grid(x_tiles_cut<T>(a.g, CB, a.cut))), block, 0, st, a);
    else
        hipLaunchKernelGGL((k_xinv_state<T, LL, PB, false>), dim3(x_grid(x_tiles(a.g, PB, false))), dim3(PB * (LL / 8)), 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t xfwd_spec_len(const XfwdArgs &a, hipStream_t st)
{
    constexpr int CB = plain_block(LL);
    dim3 grid(x_grid(x_tiles(a.g, CB, false)));
    hipLaunchKernelGGL((k_xfwd_spec<T, LL, CB>), grid, dim3(CB * (LL / 8)), 0, st, a);
    return hipGetLastError();
}

template <typename T, int MM>
hipError_t z_c2r_len(const ZArgs &a, hipStream_t st)
{
    if (z_small<MM>(a.g)) hipLaunchKernelGGL((k_z_c2r<T, MM, 1>), (ZLines<MM, 1>::grid(a.g)), dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_z_c2r<T, MM, 4>), (ZLines<MM, 4>::grid(a.g)), dim3(256), 0, st, a);
    return hipGetLastError();
}

template <typename T, int MM>
hipError_t z_r2c_len(const ZArgs &a, hipStream_t st)
{
    if (z_small<MM>(a.g)) hipLaunchKernelGGL((k_z_r2c<T, MM, 1>), (ZLines<MM, 1>::grid(a.g)), dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_z_r2c<T, MM, 4>), (ZLines<MM, 4>::grid(a.g)), dim3(256), 0, st, a);
    return hipGetLastError();
}

template <typename T, int MM, bool GIVER, bool FIVE>
hipError_t z_products_launch(const ZArgs &a, hipStream_t st)
{
    const dim3 grid = ZLines<MM, 4>::grid(a.g), block(256);
    const int fields = (GIVER ? 6 : 3) + a.ncomp;
    constexpr bool STREAM = (GIVER || FIVE) && MM >= kStreamLength / 2;
    const bool nt = STREAM && stream_bytes((size_t)fields * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    if (nt) hipLaunchKernelGGL((k_z_products<T, MM, GIVER, FIVE, STREAM, 4>), grid, block, 0, st, a);
    else if (z_small<MM>(a.g))
        hipLaunchKernelGGL((k_z_products<T, MM, GIVER, FIVE, false, 1>), (ZLines<MM, 1>::grid(a.g)), dim3(64), 0, st, a);
    else hipLaunchKernelGGL((k_z_products<T, MM, GIVER, FIVE, false, 4>), grid, block, 0, st, a);
    return hipGetLastError();
}

template <typename T, int MM>
hipError_t z_products_len(const ZArgs &a, int giver, hipStream_t st)
{
    if (giver && a.ncomp == 8) return z_products_launch<T, MM, true, true>(a, st);
    if (giver) return z_products_launch<T, MM, true, false>(a, st);
    if (a.ncomp == 5) return z_products_launch<T, MM, false, true>(a, st);
    return z_products_launch<T, MM, false, false>(a, st);
}

template <typename T, int LL, int MODE, int ST>
hipError_t x_nlin_launch(const XnlArgs &a, hipStream_t st)
{
    // One block of 512 threads fills a CU's registers (the three sums, a
    // product and the next one): 128-byte rows up to 512-point FP64 and
    // 256-point FP32 lines.  64-byte rows of 512-point FP64 lines in two blocks
    // a CU took 5041 us a launch against 4828 (before the instruction cache
    // was relieved).
    constexpr int CB = colx_block<T>(LL, 512);
    const bool nt = stream_bytes((size_t)8 * a.g.nx * a.g.ny * a.g.nzp * sizeof(cpx<T>));
    const dim3 grid(x_grid(MODE == XNL_GIVER ? x_tiles_cut<T>(a.g, CB, a.cut) : x_tiles(a.g, CB, false))), block(CB * (LL / 8));
    constexpr bool NT = LL >= kStreamLength && (ST > 0 || MODE == XNL_GIVER);
    if (NT && nt) hipLaunchKernelGGL((k_x_nlin<T, LL, CB, MODE, ST, NT>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_x_nlin<T, LL, CB, MODE, ST, false>), grid, block, 0, st, a);
    return hipGetLastError();
}

template <typename T, int LL>
hipError_t x_nlin_len(const XnlArgs &a, int mode, hipStream_t st)
{
    if (mode == XNL_GIVER) return x_nlin_launch<T, LL, XNL_GIVER, 0>(a, st);
    if (mode == XNL_TRANS) return x_nlin_launch<T, LL, XNL_TRANS, 0>(a, st);
    if (mode == XNL_SIX) return x_nlin_launch<T, LL, XNL_SIX, 0>(a, st);
    switch (a.rk.stage) {
        case 1: return x_nlin_launch<T, LL, XNL_FIVE, 1>(a, st);
        case 2: return x_nlin_launch<T, LL, XNL_FIVE, 2>(a, st);
        case 3: return x_nlin_launch<T, LL, XNL_FIVE, 3>(a, st);
        case 4: return x_nlin_launch<T, LL, XNL_FIVE, 4>(a, st);
        default: return x_nlin_launch<T, LL, XNL_FIVE, 0>(a, st);
    }
}

#define TG_KERNELS_L(N, T, P)                                                                  \
    P template hipError_t colfft_len<T, N>(const ColArgs &, int, int, hipStream_t);           \
    P template hipError_t xinv_state_len<T, N>(const XinvArgs &, hipStream_t);                \
    P template hipError_t xfwd_spec_len<T, N>(const XfwdArgs &, hipStream_t);                 \
    P template hipError_t x_nlin_len<T, N>(const XnlArgs &, int, hipStream_t);
#define TG_KERNELS_M(N, T, P)                                                                  \
    P template hipError_t z_c2r_len<T, N>(const ZArgs &, hipStream_t);                        \
    P template hipError_t z_r2c_len<T, N>(const ZArgs &, hipStream_t);                        \
    P template hipError_t z_products_len<T, N>(const ZArgs &, int, hipStream_t);

#if TG_LEN_UNIT == 0
TG_ALL_UNITS(TG_KERNELS_L, TG_KERNELS_M, extern)

template <typename T>
hipError_t launch_colfft(const Grid &g, int dir, void *const *fields, int nfields, const void *tw, hipStream_t st,
                         const Cut *cut)
{
    ColArgs a{};
    for (int i = 0; i < nfields; i++) a.f[i] = fields[i];
    a.tw = tw;
    a.nouter = g.nx;
    a.outer_stride = (long long)g.ny * g.nzp;
    a.row_stride = g.nzp;
    // the pad columns too (they hold zeros): a row's last 128-byte line is
    // written whole (257 of 264 columns written: 1903 us a launch at 512^3
    // FP64, all 264: 1780)
    a.ncol = cut ? kept_columns<T>(g, cut->z) : g.nzp;
    a.keep = cut ? cut->y : g.ny;
    TG_DISPATCH_L(T, g.ny, return (colfft_len<T, LL>)(a, dir, nfields, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_xinv_state(const Grid &g, const Band &b, double *const *V, int ncomp, void *const *U,
                             double *slots, int flags, const void *twx, hipStream_t st, double r_lo, double r_hi,
                             double a_lo, double a_hi, int dirn, const Cut *cut)
{
    XinvArgs a{};
    if (cut && !(flags & 56)) return hipErrorInvalidValue;
    a.cut = cut ? *cut : cut_none(g);
    a.r_lo = r_lo;
    a.r_hi = r_hi;
    a.a_lo = a_lo;
    a.a_hi = a_hi;
    a.dirn = dirn;
    for (int i = 0; i < ncomp; i++) { a.V[i] = V[i]; a.U[i] = U[i]; }
    a.slots = slots;
    a.tw = twx;
    a.g = g;
    a.b = b;
    a.ncomp = ncomp;
    a.flags = flags;
    TG_DISPATCH_L(T, g.nx, return (xinv_state_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_xfwd_spec(const Grid &g, void *const *W, int ncomp, double *const *out, double scale,
                            const void *twx, hipStream_t st)
{
    XfwdArgs a{};
    for (int i = 0; i < ncomp; i++) { a.W[i] = W[i]; a.out[i] = out[i]; }
    a.tw = twx;
    a.g = g;
    a.scale = scale;
    a.ncomp = ncomp;
    TG_DISPATCH_L(T, g.nx, return (xfwd_spec_len<T, LL>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_z_c2r(const Grid &g, void *const *W, int ncomp, double *const *R, const void *twm, const void *twn,
                        hipStream_t st)
{
    ZArgs a{};
    for (int i = 0; i < ncomp; i++) { a.in[i] = W[i]; a.out[i] = R[i]; }
    a.twm = twm;
    a.twn = twn;
    a.g = g;
    a.ncomp = ncomp;
    TG_DISPATCH_M(T, g.nz / 2, return (z_c2r_len<T, MM>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_z_r2c(const Grid &g, const double *const *R, int ncomp, void *const *W, const void *twm,
                        const void *twn, hipStream_t st)
{
    ZArgs a{};
    for (int i = 0; i < ncomp; i++) { a.in[i] = (void *)R[i]; a.out[i] = W[i]; }
    a.twm = twm;
    a.twn = twn;
    a.g = g;
    a.ncomp = ncomp;
    TG_DISPATCH_M(T, g.nz / 2, return (z_r2c_len<T, MM>)(a, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_z_products(const Grid &g, void *const *U, void *const *P, int giver, const void *twm,
                             const void *twn, hipStream_t st, void *const *tape, const Cut *in_u, const Cut *in_w,
                             const Cut *out)
{
    ZArgs a{};
    if ((in_u || in_w || out) && giver != 1) return hipErrorInvalidValue;
    a.lim_u = in_u ? kept_columns<T>(g, in_u->z) : g.nzp;
    a.lim_w = in_w ? kept_columns<T>(g, in_w->z) : g.nzp;
    a.lim_out = out ? kept_columns<T>(g, out->z) : g.nzp;
    // giver 2: the NS form with the five trace-shifted products; 3: the giver
    // form with the eight trace-shifted ones (MHD stage)
    a.ncomp = giver == 2 ? 5 : (giver == 3 ? 8 : (giver == 1 ? 9 : 6));
    giver = giver == 1 || giver == 3;
    if (tape && !giver)
        for (int i = 0; i < 3; i++) a.tape[i] = tape[i];
    for (int i = 0; i < (giver ? 6 : 3); i++) a.in[i] = U[i];
    for (int i = 0; i < a.ncomp; i++) a.out[i] = P[i];
    a.twm = twm;
    a.twn = twn;
    a.g = g;
    TG_DISPATCH_M(T, g.nz / 2, return (z_products_len<T, MM>)(a, giver, st));
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_x_nlin(const Grid &g, const Band &b, const RkParams &rk, void *const *P, double *const *V,
                         double *const *acc, void *const *U, const double *slots_in, double *slots_out,
                         double *const *out, const void *twx, hipStream_t st, const Cut *cut)
{
    XnlArgs a{};
    if (cut && rk.stage != -1) return hipErrorInvalidValue;
    a.cut = cut ? *cut : cut_none(g);
    // rk.stage -1: giver form, -2: transposed giver form (nonlinear term only)
    const int giver = rk.stage == -1 ? 1 : (rk.stage == -2 ? 2 : 0);
    for (int i = 0; i < (giver ? 9 : 6); i++) a.P[i] = P[i];
    for (int i = 0; i < 3; i++) {
        a.V[i] = V ? V[i] : nullptr;
        a.acc[i] = acc ? acc[i] : nullptr;
        a.U[i] = U ? U[i] : nullptr;
        a.out[i] = out ? out[i] : nullptr;
    }
    a.slots_in = slots_in;
    a.slots_out = slots_out;
    a.tw = twx;
    a.g = g;
    a.b = b;
    if (b.kind == 1) a.b.force = const_cast<double *>(slots_in);
    a.rk = rk;
    if (giver) {
        a.rk.stage = 0;
        a.rk.write_rhs = 0;
    }
    const int mode = giver == 1 ? XNL_GIVER : (giver == 2 ? XNL_TRANS : (rk.trace_free ? XNL_FIVE : XNL_SIX));
    if (mode != XNL_FIVE && a.rk.stage > 0) return hipErrorInvalidValue;
    TG_DISPATCH_L(T, g.nx, return (x_nlin_len<T, LL>)(a, mode, st));
    return hipErrorInvalidValue;
}

hipError_t launch_reality(const Grid &g, double *const *V, int ncomp, hipStream_t st)
{
    PlaneArgs a{};
    for (int i = 0; i < ncomp; i++) a.V[i] = V[i];
    a.g = g;
    a.ncomp = ncomp;
    const int n = g.nx * g.ny;
    hipLaunchKernelGGL(k_reality, dim3((n + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_dealias(const Grid &g, double *const *V, int ncomp, hipStream_t st)
{
    PlaneArgs a{};
    for (int i = 0; i < ncomp; i++) a.V[i] = V[i];
    a.g = g;
    a.ncomp = ncomp;
    hipLaunchKernelGGL(k_dealias, dim3(2048), dim3(256), 0, st, a);
    return hipGetLastError();
}

#define TG_INST(T)                                                                                              \
    template hipError_t launch_colfft<T>(const Grid &, int, void *const *, int, const void *, hipStream_t,      \
                                         const Cut *);                                                         \
    template hipError_t launch_xinv_state<T>(const Grid &, const Band &, double *const *, int, void *const *,   \
                                             double *, int, const void *, hipStream_t, double, double, double, \
                                             double, int, const Cut *);                                                     \
    template hipError_t launch_xfwd_spec<T>(const Grid &, void *const *, int, double *const *, double,          \
                                            const void *, hipStream_t);                                        \
    template hipError_t launch_z_c2r<T>(const Grid &, void *const *, int, double *const *, const void *,        \
                                        const void *, hipStream_t);                                            \
    template hipError_t launch_z_r2c<T>(const Grid &, const double *const *, int, void *const *, const void *,  \
                                        const void *, hipStream_t);                                            \
    template hipError_t launch_z_products<T>(const Grid &, void *const *, void *const *, int, const void *,     \
                                             const void *, hipStream_t, void *const *, const Cut *, const Cut *, \
                                             const Cut *);                        \
    template hipError_t launch_x_nlin<T>(const Grid &, const Band &, const RkParams &, void *const *,           \
                                         double *const *, double *const *, void *const *, const double *,      \
                                         double *, double *const *, const void *, hipStream_t, const Cut *);

TG_INST(double)
TG_INST(float)
#else
TG_THIS_UNIT(TG_KERNELS_L, TG_KERNELS_M)
#endif  // TG_LEN_UNIT

}  // namespace tg
