// tg_pass.h -- device helpers shared by the x, y and z passes (column tiles of
// the x pass, z-line real<->complex transforms, wavenumbers and the dealias
// mask) and the size dispatch of the launchers.
#pragma once
#include "tg_device.h"
#include "tg_kernels.h"

namespace tg {

// Whether a pass over `bytes` of fields streams past the 256 MiB memory-side
// cache, so that nothing it writes is still there for the next pass.
inline bool stream_bytes(size_t bytes) { return bytes > ((size_t)256 << 20); }
// Shortest x and y lines with non-temporal instances (shorter ones only stream
// that much on grids of very unequal sides).
static constexpr int kStreamLength = 64;

__device__ __forceinline__ int kwave(int l, int n) { return l <= n / 2 ? l : l - n; }

__device__ __forceinline__ bool dealias_zero(const Grid &g, int lx, int ly, int lz)
{
    if (g.basis == 1) {
        // SFF_PENCIL::Dealias (SFF_pencil_basic.cc:94-97): lx in [2Nx/3+1, Nx-1],
        // ly in [Ny/3+1, 2Ny/3-1], lz in [Nz/3+1, Nz/2] (empty y/z ranges
        // clamped); the 2/3 mode zeroes lx > 2Nx/3, |ky| > Ny/3, lz > Nz/3.
        if (g.dealias == 1) {
            int ylo = g.ny / 3 + 1, yhi = 2 * g.ny / 3 - 1;
            if (yhi < ylo) yhi = ylo;
            int zlo = g.nz / 3 + 1, zhi = g.nz / 2;
            if (zhi < zlo) zhi = zlo;
            return lx >= 2 * g.nx / 3 + 1 && (ly >= ylo && ly <= yhi) && (lz >= zlo && lz <= zhi);
        }
        if (g.dealias == 2) return lx > 2 * g.nx / 3 || abs(kwave(ly, g.ny)) > g.ny / 3 || lz > g.nz / 3;
        return false;
    }
    if (g.dealias == 1) {
        // FFF_PENCIL::Dealias (FFF_pencil_basic.cc:87-90) via Assign_sub_array
        // (:228-259): intersection of lx in [Nx/3+1, 2Nx/3-1],
        // ly in [Ny/3+1, 2Ny/3-1], lz in [Nz/3+1, Nz/2]; an empty y/z range is
        // clamped to its first index.
        int ylo = g.ny / 3 + 1, yhi = 2 * g.ny / 3 - 1;
        if (yhi < ylo) yhi = ylo;
        int zlo = g.nz / 3 + 1, zhi = g.nz / 2;
        if (zhi < zlo) zhi = zlo;
        return (lx >= g.nx / 3 + 1 && lx <= 2 * g.nx / 3 - 1) && (ly >= ylo && ly <= yhi) && (lz >= zlo && lz <= zhi);
    }
    if (g.dealias == 2) {
        int kx = abs(kwave(lx, g.nx)), ky = abs(kwave(ly, g.ny));
        return kx > g.nx / 3 || ky > g.ny / 3 || lz > g.nz / 3;
    }
    return false;
}

// The rows lx of column (ly, lz) that dealias_zero zeroes: x0 <= lx <= x1
// (x0 > x1: none).  |kx| > n/3 is n/3 < lx < n - n/3.
__device__ __forceinline__ void dealias_rows(const Grid &g, int ly, int lz, int &x0, int &x1)
{
    x0 = 1;
    x1 = 0;
    if (g.dealias == 1) {
        const int ylo = g.ny / 3 + 1, yhi = max(2 * g.ny / 3 - 1, ylo);
        const int zlo = g.nz / 3 + 1, zhi = max(g.nz / 2, zlo);
        if (ly >= ylo && ly <= yhi && lz >= zlo && lz <= zhi) {
            x0 = g.basis == 1 ? 2 * g.nx / 3 + 1 : g.nx / 3 + 1;
            x1 = g.basis == 1 ? g.nx - 1 : 2 * g.nx / 3 - 1;
        }
    } else if (g.dealias == 2) {
        const bool all = abs(kwave(ly, g.ny)) > g.ny / 3 || lz > g.nz / 3;
        x0 = all ? 0 : (g.basis == 1 ? 2 * g.nx / 3 + 1 : g.nx / 3 + 1);
        x1 = all || g.basis == 1 ? g.nx - 1 : g.nx - g.nx / 3 - 1;
    }
}

// K^(q-2) = (K^2)^((q-2)/2) of the hyperviscous factor exp((f + fh K^(q-2)) K^2)
// (Array_exp_ksqr, universal_basic.cc:265-291), integer division (q = 4: K^2),
// by repeated multiplication; q = 0 (none): 1.
__device__ __forceinline__ double hyper_power(int q, double ks)
{
    const int n = q == 0 ? 0 : (q == 4 ? 1 : (q - 2) / 2);
    double kp = 1.0;
#pragma unroll 1
    for (int i = 0; i < n; i++) kp *= ks;
    return kp;
}

// Columns of a ColX tile of L-point lines, a power of two: rows of 128 bytes (8
// FP64 or 16 FP32 columns), more where a block would have less than a
// wavefront, fewer where it would pass `threads`.
template <typename T>
__host__ __device__ constexpr int colx_block(int L, int threads)
{
    const int tpl = L / 8;
    int cb = 128 / (int)sizeof(cpx<T>);
    while (cb * tpl < 64) cb *= 2;
    while (cb > 1 && cb * tpl > threads) cb /= 2;
    return cb;
}

template <typename A, typename B>
__device__ __forceinline__ cpx<A> cvt(cpx<B> v) { return mk<A>((A)v.x, (A)v.y); }

// Lawson stage ST of one mode: the accumulator ac (stage 4: the new state),
// the next stage input vn; E = exp(-nu K^2 dt/2), stage 4 exp(-nu K^2 dt), E1
// (stage 1) exp(-nu K^2 dt).
template <int ST>
__device__ __forceinline__ void lawson(const cpx<double> &v0in, const cpx<double> &r, double E, double E1, double dt,
                                       cpx<double> &ac, cpx<double> &vn)
{
    const double c_half = 0.5 * dt, c_one = 1.0 * dt;
    const double c_sixth = (1.0 / 6) * dt, c_third = (1.0 / 3) * dt;
    if constexpr (ST == 1) {
        ac = c_sixth * (E1 * r);
        vn = E * (v0in + c_half * r);
    } else if constexpr (ST == 2) {
        ac = ac + c_third * (E * r);
        vn = E * v0in + c_half * r;
    } else if constexpr (ST == 3) {
        ac = ac + c_third * (E * r);
        vn = E * (E * v0in + c_one * r);
    } else {
        ac = ac + c_sixth * r;
        vn = E * v0in + ac;
        ac = vn;
    }
}

// Tiles of the x pass.  Work fields store each ky row of kz with the padded
// stride nzp (a multiple of 128 bytes); the FP64 state in the boundary layout
// uses nzc = Nz/2+1.  A tile is CB consecutive columns of the padded (ly,lz)
// space (pad columns lz >= nzc carry zeros), or -- patch tiles -- the kz = 0
// and kz = Nz/2 columns of every ky.
//
// Blocks are dispatched to the 8 XCDs round-robin; xcd_tile() hands each XCD
// a contiguous range of tiles so that neighbouring tiles (which share the
// 128-byte lines of the unpadded state rows) run on the same L2.
__device__ __forceinline__ int xcd_tile(int b, int nb)
{
    const int per = nb / 8;
    return (b % 8) * per + b / 8;
}

__host__ __device__ inline int x_tiles(const Grid &g, int CB, bool patch)
{
    return patch ? (2 * g.ny + CB - 1) / CB : (g.ny * g.nzp + CB - 1) / CB;
}

// Tiles of the columns that a cut keeps, and the place of one of them among
// all tiles.  Tiles wider than a row's 128-byte lines are not cut.
template <typename T>
__host__ __device__ inline int x_tiles_cut(const Grid &g, int CB, const Cut &c)
{
    if (CB * (int)sizeof(cpx<T>) > 128) return x_tiles(g, CB, false);
    return kept(g.ny, c.y) * (kept_columns<T>(g, c.z) / CB);
}
template <typename T>
__device__ __forceinline__ int x_tile_cut(const Grid &g, int CB, const Cut &c, int tile)
{
    if (CB * (int)sizeof(cpx<T>) > 128) return tile;
    const int per = kept_columns<T>(g, c.z) / CB;
    return kept_index(tile / per, g.ny, c.y) * (g.nzp / CB) + tile % per;
}

__host__ inline int x_grid(int ntiles) { return 8 * ((ntiles + 7) / 8); }

// ---------------------------------------------------------------------------
// Column tiles of the x passes that hold their points in registers (ColX).
// ---------------------------------------------------------------------------
// Keeps loads and stores on their side of it (no wait): without it the loads of
// all the later products move up to the first one and spill.
__device__ __forceinline__ void pin_memory_order()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// A value formed at this point: the sums and factors below would otherwise be
// moved to their uses (inside a later branch) and everything that they are
// formed from kept in registers until then (1.3 KB a lane spilled).
__device__ __forceinline__ void settle(double &x) { asm volatile("" : "+v"(x)); }
template <typename T>
__device__ __forceinline__ void settle(cpx<T> &z) { asm volatile("" : "+v"(z.x), "+v"(z.y)); }

// An index hidden from loop-invariant code motion: the twiddles, wavenumbers
// and LDS addresses formed from it are formed again at each use instead of
// staying in registers over the whole kernel (the twiddles alone are 56).
__device__ __forceinline__ int hidden(int j)
{
    asm volatile("" : "+v"(j));
    return j;
}

// A global address that is the same for the whole wavefront, in scalar
// registers (the sum of a field's base, a row and a thread's offset would
// otherwise be formed the other way round: a 64-bit vector address for each
// row).
typedef __attribute__((address_space(1))) char gchar;
__device__ __forceinline__ gchar *uniform_address(const void *p)
{
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return (gchar *)(((uint64_t)hi << 32) | lo);
}

// This thread's 8 points of a column (ColX order): rows j + TPL s.  p is the
// same for the whole block (its first row and column), off this thread's byte
// offset from it (under 4 GB: an eighth of a field), so that an address is a
// scalar base and one 32-bit register however many rows and fields there are.
template <bool NT, typename T>
__device__ __forceinline__ void col_load(cpx<T> *v, const cpx<T> *p, size_t step, uint32_t off)
{
    typedef __attribute__((address_space(1))) const vec2<T> gvec;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        gvec *q = (gvec *)(uniform_address(p + s * step) + off);
        vec2<T> x;
        if constexpr (NT) x = __builtin_nontemporal_load(q);
        else x = *q;
        v[s] = mk<T>(x.x, x.y);
    }
}
template <bool NT, typename T>
__device__ __forceinline__ void col_store(const cpx<T> *v, cpx<T> *p, size_t step, uint32_t off)
{
    typedef __attribute__((address_space(1))) vec2<T> gvec;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        gvec *q = (gvec *)(uniform_address(p + s * step) + off);
        vec2<T> x;
        x.x = v[s].x;
        x.y = v[s].y;
        if constexpr (NT) __builtin_nontemporal_store(x, q);
        else *q = x;
    }
}

// The CB columns of a block of an x pass, thread t on column t % CB at rows
// t / CB + TPL s.  Tiles of at most 128-byte rows divide nzp and lie within one
// ky row, the same for the whole block; the wider ones of short lines do not,
// and the last one may run past the last column (those threads move the last
// column and store nothing).  Columns of the work fields (padded layout, T or
// FP64) are at base + cw0 with byte offsets offt / offw and row step stepw, of
// the state (boundary layout, FP64) at base + state0 with offs and steps.
template <typename T, int L, int CB>
struct ColTile {
    static constexpr int TPL = L / 8;
    static constexpr bool WIDE = CB * sizeof(cpx<T>) > 128;
    int c, j, ly, lz, lz0, cw0;
    bool inside, live;   // a column of the tile; one that holds modes (pad columns carry zeros)
    size_t stepw, steps, state0;
    uint32_t offt, offw, offs;

    // patch: the kz = 0 and Nz/2 columns of every ky (bases at the fields' start)
    __device__ __forceinline__ ColTile(const Grid &g, int tile, bool patch = false)
    {
        c = threadIdx.x % CB;
        j = threadIdx.x / CB;
        const int ncol = g.ny * g.nzp;
        if (patch) {
            const int p = tile * CB + c, q = min(p, 2 * g.ny - 1);
            inside = live = p < 2 * g.ny;
            ly = q >> 1;
            lz = q & 1 ? g.nz / 2 : 0;
            lz0 = cw0 = 0;
            state0 = 0;
            stepw = (size_t)TPL * ncol;
            steps = (size_t)TPL * g.ny * g.nzc;
            const uint32_t cw = (uint32_t)((size_t)j * ncol + ly * g.nzp + lz);
            offt = cw * (uint32_t)sizeof(cpx<T>);
            offw = cw * 16u;
            offs = (uint32_t)((size_t)j * g.ny * g.nzc + ly * g.nzc + lz) * 16u;
            return;
        }
        cw0 = tile * CB;
        const int cwt = WIDE ? min(cw0 + c, ncol - 1) : cw0;
        inside = !WIDE || cw0 + c < ncol;
        ly = cwt / g.nzp;
        lz0 = WIDE ? 0 : cwt % g.nzp;
        lz = WIDE ? cwt % g.nzp : lz0 + c;
        live = inside && lz < g.nzc;
        const size_t ncw = (size_t)ncol, ncs = (size_t)g.ny * g.nzc;
        stepw = (size_t)TPL * ncw;
        steps = (size_t)TPL * ncs;
        state0 = WIDE ? 0 : (size_t)ly * g.nzc + min(lz0, g.nzc - 1);
        const uint32_t colt = WIDE ? cwt - cw0 : c;
        offt = (uint32_t)(j * ncw + colt) * (uint32_t)sizeof(cpx<T>);
        offw = (uint32_t)(j * ncw + colt) * 16u;
        // (a pad column reads the last one; a tile may hold pad columns only)
        offs = (uint32_t)(j * ncs + (WIDE ? ly * g.nzc + min(lz, g.nzc - 1) : max(min(c, g.nzc - 1 - lz0), 0))) * 16u;
    }
};

// the slot of a mode, -1 outside the box
__device__ __forceinline__ int band_slot(const Band &b, int kx, int ky, int kz)
{
    if (abs(kx) > b.h[0] || abs(ky) > b.h[1] || kz > b.h[2]) return -1;
    return ((kx + b.h[0]) * (2 * b.h[1] + 1) + (ky + b.h[1])) * (b.h[2] + 1) + kz;
}

__device__ __forceinline__ double kmag(const Grid &g, int kx, int ky, int kz)
{
    const double a = kx * g.kf[0], b = ky * g.kf[1], c = kz * g.kf[2];
    return sqrt(a * a + b * b + c * c);
}

__device__ __forceinline__ bool in_band(const Grid &g, const Band &b, int kx, int ky, int kz)
{
    const double K = kmag(g, kx, ky, kz);
    return K > b.r_in && K <= b.r_out;
}

// ---------------------------------------------------------------------------
// z-line transforms.  A real line x[0..N) (N = 2M) is packed as
// z[n] = x[2n] + i x[2n+1]; a complex line holds X[0..M].
// c2r: Z'[k] = (X[k] + conj X[M-k]) + i W^-k (X[k] - conj X[M-k]), with the
//      imaginary parts of X[0], X[M] dropped; z = IDFT_M(Z') (unscaled), so
//      x = sum_k X_herm[k] e^{+2 pi i k n / N}.
// r2c: Z = DFT_M(z); X[k] = ((Z[k] + conj Z[M-k]) - i W^k (Z[k] - conj Z[M-k]))/2.
// W = exp(-2 pi i / N); twn holds W^k for k = 0..M.
// ---------------------------------------------------------------------------
// The twiddles of a z kernel in LDS (2 M entries: m in pass order, then n): read
// from global memory between two lines' stores, each would wait for the stores
// before it (loads and stores retire in order).
template <typename T, int M>
struct ZTwiddles {
    const cpx<T> *m, *n;
    // all threads of the block; ends in a barrier
    __device__ __forceinline__ ZTwiddles(cpx<T> *lds, const void *twm, const void *twn) : m(lds), n(lds + M)
    {
        for (int i = threadIdx.x; i < M; i += blockDim.x) {
            lds[i] = ((const cpx<T> *)twm)[i];
            lds[M + i] = ((const cpx<T> *)twn)[i];
        }
        lds_barrier();
    }
};

// The M+1 points of a complex line: v[s] = X[j + TPL*s], xm = X[M] (read by
// every thread of the line; member-wise copies keep v in registers).
// LIM: the points from lim on are zero and not read.
template <typename T, int M, bool NT = false, bool LIM = false>
__device__ __forceinline__ void zline_load(cpx<T> *v, cpx<T> &xm, const cpx<T> *__restrict__ X, int j, int lim = 0)
{
    constexpr int TPL = M / 8;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        v[s] = mk<T>(0, 0);
        if (!LIM || j + TPL * s < lim) v[s] = gload<NT>(X + j + TPL * s);
    }
    xm = mk<T>(0, 0);
    if (!LIM || M < lim) xm = gload<false>(X + M);
}

// c2r of a line already loaded by zline_load (v in, samples out in v).
template <typename T, int M>
__device__ __forceinline__ void zline_c2r_from(cpx<T> *v, cpx<T> xm, cpx<T> *lds, const ZTwiddles<T, M> &tw, int j)
{
    constexpr int TPL = M / 8;
    // the line (M+1 points) in LDS, for the mirrored points
#pragma unroll
    for (int s = 0; s < 8; s++) lds[lpad(j + TPL * s)] = mk<T>(v[s].x, v[s].y);
    if (j == 0) lds[lpad(M)] = xm;
    line_sync();
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = j + TPL * s;
        cpx<T> xk = v[s];
        cpx<T> xm = lds[lpad(M - k)];
        if (k == 0) { xk.y = 0; xm.y = 0; }
        const cpx<T> a = xk + conj(xm);
        const cpx<T> d = xk - conj(xm);
        const cpx<T> w = tw.n[k];  // W^k ; we need W^-k = conj(w)
        const cpx<T> e = mk<T>(d.x * w.x + d.y * w.y, d.y * w.x - d.x * w.y);
        v[s] = a + mk<T>(-e.y, e.x);
    }
    line_sync();
    fft_line<M, +1>(v, lds, tw.m, j);
}

template <typename T, int M, bool NT = false, bool LIM = false>
__device__ __forceinline__ void zline_c2r(cpx<T> *v, const cpx<T> *__restrict__ X, cpx<T> *lds,
                                          const ZTwiddles<T, M> &tw, int j, int lim = 0)
{
    cpx<T> xm;
    zline_load<T, M, NT, LIM>(v, xm, X, j, lim);
    zline_c2r_from<T, M>(v, xm, lds, tw, j);
}

// The line's npad = nzp - M entries from X[M] on are written too (zeros after
// X[M]): whole 128-byte lines.  LIM: only the points before lim are written.
template <typename T, int M, bool NT = false, bool LIM = false>
__device__ __forceinline__ void zline_r2c_post(cpx<T> *v, cpx<T> *__restrict__ X, cpx<T> *lds,
                                               const ZTwiddles<T, M> &tw, int j, bool store, int npad, int lim = 0)
{
    constexpr int TPL = M / 8;
    fft_line<M, -1>(v, lds, tw.m, j);
#pragma unroll
    for (int s = 0; s < 8; s++) lds[lpad(j + TPL * s)] = v[s];
    line_sync();
    const T h = (T)0.5;
    const cpx<T> z0 = lds[0];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int k = j + TPL * s;
        const cpx<T> zk = v[s];
        const cpx<T> zm = lds[lpad(k == 0 ? 0 : M - k)];
        const cpx<T> a = zk + conj(zm);
        const cpx<T> d = zk - conj(zm);
        const cpx<T> w = tw.n[k];
        const cpx<T> e = d * w;  // W^k d
        if (store && (!LIM || k < lim)) gstore<NT>(X + k, mk<T>(h * (a.x + e.y), h * (a.y - e.x)));
    }
    if (store && (!LIM || M < lim))
        for (int i = j; i < npad; i += TPL) gstore<NT>(X + M + i, mk<T>(i == 0 ? z0.x - z0.y : (T)0, (T)0));
    line_sync();
}

struct ZArgs {
    void *in[6];
    void *out[9];
    void *tape[3];  // optional: real-space velocity lines (Nx*Ny lines of Nz/2 packed points)
    const void *twm, *twn;
    Grid g;
    int ncomp;
    int lim_u, lim_w, lim_out;  // giver form: columns of the fields and products that are dealt with
};

// The lines of a block of a z pass: M/8 threads a line, as many lines a wavefront
// as fit (of the lengths with factors 3 and 5 a few lanes are left over: with
// their lines across wavefronts, behind block barriers, the products of a
// 240 x 160 x 96 FP64 step took 96 us, now 87), W wavefronts.
template <int M, int W>
struct ZLines {
    static constexpr int TPL = M / 8, LPW = 64 / TPL, LPB = LPW * W, THREADS = 64 * W;
    static_assert(TPL <= 64, "a z line lies in one wavefront");
    int li, j;
    bool spare;   // a lane without a line (it ends after the last block barrier)
    size_t line, safe;
    bool valid;
    __device__ __forceinline__ ZLines(const Grid &g)
    {
        const int lane = threadIdx.x & 63, l = lane / TPL;
        if constexpr (64 % TPL == 0) {
            spare = false;
            li = threadIdx.x / TPL;
            j = threadIdx.x % TPL;
        } else {
            spare = l >= LPW;
            li = (threadIdx.x / 64) * LPW + (l < LPW ? l : LPW - 1);
            j = lane % TPL;
        }
        line = (size_t)blockIdx.x * LPB + li;
        const size_t n = (size_t)g.nx * g.ny;
        valid = line < n;
        safe = valid ? line : n - 1;
    }
    static dim3 grid(const Grid &g) { return dim3((unsigned)(((size_t)g.nx * g.ny + LPB - 1) / LPB)); }
};
// Blocks of one wavefront where blocks of four would leave CUs idle: 64 of them
// at 64^3 FP64, 19.8 us a launch of the products against 15.8; with two a CU and
// more (128^3 and larger) nothing changes.
template <int M>
inline bool z_small(const Grid &g) { return (size_t)g.nx * g.ny < (size_t)256 * ZLines<M, 4>::LPB; }

// ---------------------------------------------------------------------------
// Transform lengths with compiled kernels, and the size dispatch of the
// launchers (lengths are compile-time).  x and y lines take L, z lines the
// half length M = Nz/2.  Power-of-two lengths in both precisions; lengths
// with radix-3/5 factors in FP64.
//
// Each launcher fills its argument block and calls a per-length function
// (NAME_len<T, L>) that launches the kernels of that length.  The per-length
// functions are instantiated in length units -- the same source compiled
// once per unit with TG_LEN_UNIT = 1..4 (1: power-of-two FP64, 2:
// power-of-two FP32, 3 and 4: radix-3/5 lengths FP64) -- so that the kernel
// instances compile in parallel; unit 0 (the plain compilation) holds the
// launchers and declares the per-length functions extern.
// ---------------------------------------------------------------------------
#define TG_L_POW2(F, T, P) F(8, T, P) F(16, T, P) F(32, T, P) F(64, T, P) F(128, T, P) F(256, T, P) F(512, T, P) \
    F(1024, T, P)
#define TG_L_ODDA(F, T, P) F(24, T, P) F(40, T, P) F(48, T, P) F(80, T, P) F(96, T, P) F(120, T, P) F(160, T, P) \
    F(192, T, P)
#define TG_L_ODDB(F, T, P) F(240, T, P) F(320, T, P) F(384, T, P) F(480, T, P) F(640, T, P) F(768, T, P) F(960, T, P)
#define TG_M_POW2(F, T, P) F(8, T, P) F(16, T, P) F(32, T, P) F(64, T, P) F(128, T, P) F(256, T, P) F(512, T, P)
#define TG_M_ODDA(F, T, P) F(24, T, P) F(40, T, P) F(48, T, P) F(80, T, P) F(96, T, P) F(120, T, P) F(160, T, P) \
    F(192, T, P)
#define TG_M_ODDB(F, T, P) F(240, T, P) F(320, T, P) F(384, T, P) F(480, T, P)

#define TG_UNIT_1(FL, FM, P) TG_L_POW2(FL, double, P) TG_M_POW2(FM, double, P)
#define TG_UNIT_2(FL, FM, P) TG_L_POW2(FL, float, P) TG_M_POW2(FM, float, P)
#define TG_UNIT_3(FL, FM, P) TG_L_ODDA(FL, double, P) TG_M_ODDA(FM, double, P)
#define TG_UNIT_4(FL, FM, P) TG_L_ODDB(FL, double, P) TG_M_ODDB(FM, double, P)
#define TG_ALL_UNITS(FL, FM, P) TG_UNIT_1(FL, FM, P) TG_UNIT_2(FL, FM, P) TG_UNIT_3(FL, FM, P) TG_UNIT_4(FL, FM, P)
#define TG_CAT_(a, b) a##b
#define TG_CAT(a, b) TG_CAT_(a, b)
// the instantiations of this compilation's length unit
#define TG_THIS_UNIT(FL, FM) TG_CAT(TG_UNIT_, TG_LEN_UNIT)(FL, FM, )
#define TG_NO_LENGTHS(N, T, P)

#ifndef TG_LEN_UNIT
#define TG_LEN_UNIT 0
#endif

#define TG_CASE_P2(N, T, CALL) \
    case N: { constexpr int LL = N, MM = N; (void)LL; (void)MM; CALL; } break;
#define TG_CASE_ODD(N, T, CALL)                        \
    case N: {                                          \
        constexpr int LL = N, MM = N;                  \
        (void)LL;                                      \
        (void)MM;                                      \
        if constexpr (sizeof(T) == 8) { CALL; }        \
        else return hipErrorInvalidValue;              \
    } break;
// CALL (no top-level commas: parenthesise template argument lists) is
// compiled once per length with the constant LL (x/y lines) or MM (z half
// lines); a length without kernels returns hipErrorInvalidValue.
#define TG_DISPATCH_L(T, Lval, CALL)                                                                  \
    switch (Lval) {                                                                                   \
        TG_L_POW2(TG_CASE_P2, T, CALL) TG_L_ODDA(TG_CASE_ODD, T, CALL) TG_L_ODDB(TG_CASE_ODD, T, CALL) \
        default: return hipErrorInvalidValue;                                                         \
    }
#define TG_DISPATCH_M(T, Mval, CALL)                                                                  \
    switch (Mval) {                                                                                   \
        TG_M_POW2(TG_CASE_P2, T, CALL) TG_M_ODDA(TG_CASE_ODD, T, CALL) TG_M_ODDB(TG_CASE_ODD, T, CALL) \
        default: return hipErrorInvalidValue;                                                         \
    }

// Host checks of a length against the compiled ones (x/y lines L, z half
// lines M; FP32 takes powers of two only).
#define TG_OK_P2(N, T, P) case N: return true;
#define TG_OK_ODD(N, T, P) case N: return !fp32;
inline bool l_compiled(int n, bool fp32)
{
    switch (n) {
        TG_L_POW2(TG_OK_P2, , ) TG_L_ODDA(TG_OK_ODD, , ) TG_L_ODDB(TG_OK_ODD, , )
        default: return false;
    }
}
inline bool m_compiled(int n, bool fp32)
{
    switch (n) {
        TG_M_POW2(TG_OK_P2, , ) TG_M_ODDA(TG_OK_ODD, , ) TG_M_ODDB(TG_OK_ODD, , )
        default: return false;
    }
}
#undef TG_OK_P2
#undef TG_OK_ODD

}  // namespace tg
