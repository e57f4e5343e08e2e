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
