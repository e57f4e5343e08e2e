"""Random forcing of wide bands: parity with the oracle, and no device memory
of its own (48 bytes a mode of the band's box would be 29 MB here)."""
import numpy as np
import pytest

import tg_oracle as to
from gpu_util import dev, host, log, rel_l2_vec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

# the parity bounds of the NS step tests: FP64 1e-12; FP32 transforms 2e-5
TOL = {api.PREC_FP64: 1e-12, api.PREC_FP32: 2e-5}


@pytest.mark.parametrize("prec", [api.PREC_FP64, api.PREC_FP32])
def test_wide_band(prec):
    N, r_out = (8, 512, 256), 400.0
    log(f"{N} {prec}")
    o = to.Oracle(N, dealias=to.DEALIAS_TWOTHIRDS, strong_reality=True)
    V = o.init_field(kind=1, k0=4.0, kmin=1.0, kmax=100.0, energy=0.5, seed=3)
    b = api.FFF_Basis(N, precision=prec, dealias=to.DEALIAS_TWOTHIRDS, strong_reality=True)
    U = api.FluidVF(b, 0.01)
    U.set_field([dev(v) for v in V])
    ta = api.Time_advance_incompress(U, 1e-3, 2, 0.2, 0.5, r_out, 0.05, 0.01, 5)
    held = b.device_bytes()
    ta.Time_advance_step(1)
    # the shells' supplies are kept: 16 bytes each
    assert b.device_bytes() - held <= 16 * (r_out + 2)
    fl = to.Fluid(0.01, 1e-3, 2, 0.2, 0.5, r_out, 0.0, 0, 0.05, 0.01, 5)
    o.rk4_step(fl, V)
    err = rel_l2_vec([host(v) for v in U.cvf], V)
    log(f"  {err:.3e}")
    assert err <= TOL[prec]
    b.close()


@pytest.mark.parametrize("prec", [api.PREC_FP64, api.PREC_FP32])
def test_calls_after_a_forced_step(prec):
    """The force lies in work fields of other calls: they give the same on a
    plan that has just made a forced step as on a new one."""
    N = (16, 32, 64)
    log(f"{N} {prec}")

    def calls(forced):
        b = api.FFF_Basis(N, precision=prec, dealias=to.DEALIAS_TWOTHIRDS, strong_reality=False)
        if forced:
            U = api.FluidVF(b, 0.01)
            U.Init_cond_spectrum(kind=0, k0=4.0, kmin=1.0, kmax=8.0, energy=0.5, seed=2)
            api.Time_advance_incompress(U, 1e-3, 2, 1e6, 0.5, 50.0, 0.0, 1e-9, 5).Time_advance_step(1)
        out = []
        for call in range(4):
            U, W = api.FluidVF(b, 0.01), api.FluidVF(b, 0.02)
            U.Init_cond_spectrum(kind=0, k0=4.0, kmin=1.0, kmax=20.0, energy=0.5, seed=3)
            W.Init_cond_spectrum(kind=0, k0=4.0, kmin=1.0, kmax=20.0, energy=0.3, seed=4)
            if call == 0:
                r = np.array([0.0, 2.0, 4.0, 7.0, np.inf])
                out += list(api.EnergyTr(b, r, r).Compute_flux_and_shell_tr(U))
            elif call == 1:
                api.Nlin_incompress.Compute_nlin(U, W)
                out += [host(a) for a in U.nlin]
            elif call == 2:
                api.Time_advance_incompress_MHD(U, W, 1e-3).Time_advance_step(1)
                out += [host(a) for a in U.cvf + W.cvf]
            else:
                ad = api.Adjoint_incompress(U, 1e-3)
                ad.Forward(2)
                out += [host(a) for a in ad.Backward([w.clone() for w in W.cvf])]
        b.close()
        return out

    for got, want in zip(calls(True), calls(False)):
        assert np.isfinite(want).all() and np.array_equal(got, want)
