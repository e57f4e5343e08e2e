// tg_chff.h -- launchers of the Chebyshev (ChFF) line kernels.
#pragma once
#include <hip/hip_runtime.h>
#include "tg_kernels.h"

namespace tg {

// Helmholtz solves per (ky, kz) column, lambda = Kperp^2 + lam_sup, wall values
// vp (x = 1) and vm (x = -1) per part (real, imaginary): of one array, R -> U
// (E = 2 complex, 1 real), or, with P, of the momentum equation's components
// comp .. comp + ncomp - 1 with right-hand side ((N - V/dt) + grad P) / (-nu),
// into V (complex).  X, Y: scratch of ny * nzc * nx doubles a component, Y
// times E (lines too long for LDS).
struct HelmArgs {
    const double *R;
    double *U;
    const double *N[3], *P;
    double *V[3];
    double *X, *Y;
    Grid g;
    double lam_sup;
    double vp[2], vm[2];
    double dt, nu;
    int E, comp;
    int pressure_switch;  // Kperp = 0 with a pressure: the linear profile
};

// Compute_pressure_Ux_chebyshev: P, V1 complex; homogeneous solutions real
struct InflArgs {
    double *P, *V1;
    const double *pp, *pm, *vxp, *vxm, *M;
    int nx, ny, nzc;
    double kf;
};

hipError_t launch_cheb_deriv(const Grid &g, const double *A, double *B, bool complex_, hipStream_t st);
hipError_t launch_helmholtz(const HelmArgs &a, hipStream_t st, int ncomp = 1);
hipError_t launch_influence(const Grid &g, const double *vxp, const double *vxm, double *M, hipStream_t st);
hipError_t launch_influence_correct(const InflArgs &a, hipStream_t st);
hipError_t launch_scale_real(double *a, size_t n, double divisor, hipStream_t st);
hipError_t launch_fill_double(double *a, size_t n, double v, hipStream_t st);

}  // namespace tg
