"""The fused NS x pass at the edges of its column tiles, against the oracle.

Short lines take tiles wider than a 128-byte row (several ky rows a tile, the
last tile past the last column), 512-point FP32 lines half rows (a tile of pad
columns only), the others one row; the forced modes come from the alpha slots
or from the random force's table, whose box may reach the Nyquist planes."""
import numpy as np
import pytest

import tg_oracle as to
from gpu_util import dev, host, log, rel_l2_vec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

# the parity bounds of the NS step tests: FP64 1e-12; FP32 transforms 2e-5
TOL = {api.PREC_FP64: 1e-12, api.PREC_FP32: 2e-5}
GRIDS = [((8, 8, 16), api.PREC_FP64), ((8, 24, 48), api.PREC_FP64), ((16, 8, 32), api.PREC_FP64), ((24, 8, 80), api.PREC_FP64),
         ((32, 16, 16), api.PREC_FP64), ((40, 8, 16), api.PREC_FP64), ((640, 8, 16), api.PREC_FP64), ((1024, 8, 16), api.PREC_FP64),
         ((8, 8, 16), api.PREC_FP32), ((16, 8, 64), api.PREC_FP32), ((64, 8, 32), api.PREC_FP32), ((512, 8, 16), api.PREC_FP32),
         ((1024, 8, 32), api.PREC_FP32)]
FORCES = {"none": (0, 0.0, 0.0, 0.0, 0.0, 0.0, 0), "alpha": (1, 0.2, 1.0, 2.5, 0.0, 0.0, 0), "random": (2, 0.2, 1.0, 3.0, 0.1, 0.01, 5),
          "random_all": (2, 0.2, 0.5, 40.0, 0.0, 0.01, 9)}


@pytest.mark.parametrize("force", sorted(FORCES))
@pytest.mark.parametrize("N,prec", GRIDS)
def test_forced_steps(N, prec, force):
    log(f"{N} {prec} {force}")
    kind, eps, r_in, r_out, hel, tau, seed = FORCES[force]
    for dealias, strong, hyper in ((to.DEALIAS_REF_CORNER, True, 0), (to.DEALIAS_TWOTHIRDS, False, 4)):
        o = to.Oracle(N, dealias=dealias, strong_reality=strong)
        V = o.init_field(kind=1, k0=4.0, kmin=1.0, kmax=max(N) / 3, energy=0.5, seed=3)
        b = api.FFF_Basis(N, precision=prec, dealias=dealias, strong_reality=strong)
        U = api.FluidVF(b, 0.01, hyper_dissipation_coefficient=1e-5 if hyper else 0.0, hyper_dissipation_exponent=hyper)
        U.set_field([dev(v) for v in V])
        api.Time_advance_incompress(U, 1e-3, kind, eps, r_in, r_out, hel, tau, seed).Time_advance_step(2)
        fl = to.Fluid(0.01, 1e-3, kind, eps, r_in, r_out, 1e-5 if hyper else 0.0, hyper, hel, tau, seed)
        o.rk4_step(fl, V)
        o.rk4_step(fl, V)
        assert all(np.isfinite(v).all() for v in V)
        assert rel_l2_vec([host(v) for v in U.cvf], V) <= TOL[prec]
        b.close()
