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
