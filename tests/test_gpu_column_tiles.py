"""The fused x passes of MHD, Rayleigh-Benard convection and the adjoint, and
the plain x passes, at the edges of their column tiles, against the oracle:
short lines (tiles wider than a 128-byte row, the last one past the last
column), a tile of pad columns only, lines with radix-3/5 factors and the
longest ones (rows of less than 128 bytes)."""
import numpy as np
import pytest

import tg_oracle as to
from gpu_util import dev, host, log, rel_l2, rel_l2_vec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

# the parity bounds of the step tests: FP64 1e-12; FP32 transforms 2e-5
TOL = {api.PREC_FP64: 1e-12, api.PREC_FP32: 2e-5}
GRIDS = [((8, 8, 16), api.PREC_FP64), ((16, 24, 48), api.PREC_FP64), ((24, 8, 32), api.PREC_FP64), ((40, 8, 80), api.PREC_FP64),
         ((640, 8, 16), api.PREC_FP64), ((1024, 8, 16), api.PREC_FP64),
         ((8, 8, 16), api.PREC_FP32), ((16, 8, 64), api.PREC_FP32), ((512, 8, 32), api.PREC_FP32), ((1024, 8, 16), api.PREC_FP32)]


@pytest.mark.parametrize("N,prec", GRIDS)
def test_mhd_steps(N, prec):
    log(f"mhd {N} {prec}")
    nu, eta, dt = 5e-3, 3e-3, 1e-3
    for dealias, strong in ((to.DEALIAS_REF_CORNER, True), (to.DEALIAS_TWOTHIRDS, False)):
        o = to.Oracle(N, dealias=dealias, strong_reality=strong)
        V = o.init_field(kind=1, kmin=1.0, kmax=max(N) / 3, energy=0.5, seed=3)
        W = o.init_field(kind=1, kmin=1.0, kmax=max(N) / 3, energy=0.25, seed=4)
        b = api.FFF_Basis(N, precision=prec, dealias=dealias, strong_reality=strong)
        U, B = api.FluidVF(b, nu), api.FluidVF(b, eta)
        U.set_field([dev(v) for v in V])
        B.set_field([dev(w) for w in W])
        api.Time_advance_incompress_MHD(U, B, dt).Time_advance_step(2)
        fl = to.Fluid(nu, dt, 0, 0, 0, 0)
        for _ in range(2):
            o.rk4_step_mhd(fl, eta, V, W)
        assert rel_l2_vec([host(v) for v in U.cvf] + [host(w) for w in B.cvf], V + W) <= TOL[prec]
        b.close()


def _spec(shape, seed, real_mean):
    """A smooth random spectrum with the conjugate symmetry left to the step."""
    r = np.random.default_rng(seed)
    k = [np.arange(shape[0]), np.minimum(np.arange(shape[1]), shape[1] - np.arange(shape[1])), np.arange(shape[2])]
    w = np.exp(-0.5 * (k[0][:, None, None] + k[1][None, :, None] + k[2][None, None, :]))
    s = 0.1 * w * (r.standard_normal(shape) + 1j * r.standard_normal(shape))
    if real_mean:
        s[0] = 0.0
    return s


@pytest.mark.parametrize("N,prec", [g for g in GRIDS if g[0][0] <= 640])
def test_rbc_steps(N, prec):
    log(f"rbc {N} {prec}")
    for dealias, reality in ((to.DEALIAS_REF_CORNER, 2), (to.DEALIAS_TWOTHIRDS, 0)):
        o = to.Oracle(N, kfactor=(np.pi, 1.5, 1.0), dealias=dealias, strong_reality=False)
        V = [_spec(o.cshape, 50 + c, c == 0) for c in range(3)]
        T = _spec(o.cshape, 53, True)
        b = api.SFF_Basis(N, kfactor=(np.pi, 1.5, 1.0), precision=prec, dealias=dealias, reality=reality)
        U, S = api.FluidVF(b), api.FluidSF(b)
        U.set_field([dev(v) for v in V])
        S.set_field(dev(T))
        api.Time_advance_incompress_RBC(U, S, 1e4, 1.0, 1e-5).Time_advance_step(2)
        for _ in range(2):
            o.rk4_step_rbc(to.Rbc(1e4, 1.0, 1e-5, reality), V, T)
        # the long lines' x-derivatives multiply round-off by K_max = pi L
        tol = TOL[prec] * max(1.0, (np.pi * N[0] / 1000.0) ** 2)
        assert rel_l2_vec([host(v) for v in U.cvf] + [host(S.F)], V + [T]) <= tol
        b.close()


@pytest.mark.parametrize("N,prec", GRIDS)
def test_adjoint_sweep(N, prec):
    """Two forward steps and the sweep back: each mode of the fused x pass."""
    log(f"adjoint {N} {prec}")
    o = to.Oracle(N, dealias=to.DEALIAS_REF_CORNER, strong_reality=False)
    V = o.init_field(kind=1, kmin=1.0, kmax=max(N) / 3, energy=0.5, seed=41)
    r_lo, r_hi = 0.5, 5.0
    loss_ref, grad_ref = o.adjoint_shell_energy(to.Fluid(0.01, 1e-3, 0, 0.0, 0.0, 0.0), V, 2, r_lo, r_hi)
    b = api.FFF_Basis(N, precision=prec, strong_reality=False)
    U = api.FluidVF(b, 0.01)
    U.set_field([dev(v) for v in V])
    adj = api.Adjoint_incompress(U, 1e-3)
    adj.Forward(2)
    k = [np.minimum(np.arange(n), n - np.arange(n)) for n in N[:2]] + [np.arange(N[2] // 2 + 1)]
    K = np.sqrt(k[0][:, None, None] ** 2.0 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2)
    # the oracle's loss: the energy of the shell, the kz = 0 plane at half weight
    m = ((K >= r_lo) & (K < r_hi)).astype(np.float64)
    m[:, :, 0] *= 0.5
    m = torch.as_tensor(m, device="cuda")
    lam = [2.0 * m * v for v in U.cvf]
    adj.Backward(lam)
    # the bounds of the gradient tests: 1e-11, FP32 transforms 2e-5
    assert rel_l2_vec([host(x) for x in lam], grad_ref) <= (1e-11 if prec == api.PREC_FP64 else 2e-5)
    b.close()


@pytest.mark.parametrize("N,prec", GRIDS)
def test_transforms_keep_and_drop_modes(N, prec):
    """The plain x passes on a random spectrum: transforms, the shell filter of
    the transfer functions (columns without a mode to keep are not read)."""
    log(f"transforms {N} {prec}")
    tol = 1e-12 if prec == api.PREC_FP64 else 1e-5
    o = to.Oracle(N)
    b = api.FFF_Basis(N, precision=prec)
    r = np.random.default_rng(1).standard_normal(o.rshape)
    r[:, :, -2:] = 0.0
    A, Ar = b.complex_array(), b.real_array()
    b.Forward_transform(dev(r), A)
    b.Inverse_transform(A, Ar)
    assert rel_l2(host(A), o.forward(r)) <= tol and rel_l2(host(Ar), r) <= tol
    if prec == api.PREC_FP32:
        b.close()
        return
    V = o.init_field(kind=1, kmin=1.0, kmax=max(N) / 3, energy=0.5, seed=7)
    radii = np.array([0.0, 1.5, 3.0, np.inf])
    U = api.FluidVF(b)
    U.set_field([dev(v) for v in V])
    got = api.EnergyTr(b, radii, radii).Compute_shell_tr(U)
    want = o.shell_to_shell([v.copy() for v in V], radii)
    assert rel_l2(got, want) <= 1e-11
    b.close()


@pytest.mark.parametrize("N,prec,kf", [((64, 24, 48), api.PREC_FP64, (1.0, 1.0, 1.0)), ((120, 40, 80), api.PREC_FP64, (1.0, 2.0, 0.5)),
                                       ((32, 16, 16), api.PREC_FP64, (1.0, 1.0, 1.0)), ((64, 16, 128), api.PREC_FP64, (1.0, 1.0, 1.0)),
                                       ((128, 32, 64), api.PREC_FP32, (1.0, 1.0, 1.0))])
def test_transfers_of_cut_fields(N, prec, kf):
    """Flux, shell and ring transfers only form the modes that the 2/3 rule and
    the giver's radius keep; without the rule, the giver's radius alone."""
    log(f"cut transfers {N} {prec} {kf}")
    # FP64 as the other transfer tests; FP32 products round at 1e-7 of a term, the sums cancel some digits
    tol = 1e-11 if prec == api.PREC_FP64 else 1e-4
    for dealias in (to.DEALIAS_TWOTHIRDS, to.DEALIAS_REF_CORNER):
        o = to.Oracle(N, kfactor=kf, dealias=dealias)
        V = o.init_field(kind=1, kmin=0.5, kmax=max(N), energy=0.5, seed=9)
        b = api.FFF_Basis(N, kfactor=kf, precision=prec, dealias=dealias)
        U = api.FluidVF(b)
        U.set_field([dev(v) for v in V])
        radii = np.array([0.0, 0.75, 2.0, 5.0, 9.0, np.inf])
        # work buffers of an earlier call hold what they like
        b.Inverse_transform(dev(np.full(o.cshape, 1e200 + 0j)), b.real_array())
        et = api.EnergyTr(b, radii, radii)
        flux, S = et.Compute_flux_and_shell_tr(U)
        assert rel_l2(S, o.shell_to_shell([v.copy() for v in V], radii)) <= tol
        assert rel_l2(flux, o.flux([v.copy() for v in V], radii)) <= tol
        assert rel_l2(et.Compute_flux(U), o.flux([v.copy() for v in V], radii)) <= tol
        b.close()
