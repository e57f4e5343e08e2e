"""The Chebyshev line kernels over the range of line lengths: the shortest, the
last whose recurrences fit LDS and the first that do not, lines with radix-3/5
factors, several wavefronts of threads a column, and column counts that leave
blocks partly empty."""
import numpy as np
import pytest

import tg_oracle as to
from gpu_util import dev, host, log, rel_l2, rel_l2_vec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

KF = (1.0, 0.5, 2.0)


@pytest.mark.parametrize("N", [(8, 8, 16), (16, 24, 48), (24, 8, 16), (80, 8, 16), (96, 8, 32), (256, 8, 16), (512, 8, 16)])
def test_chff_lines(N):
    log(f"chff {N}")
    o = to.Oracle(N, kfactor=KF, dealias=to.DEALIAS_NONE, strong_reality=False)
    rng = np.random.default_rng(60)
    damp = np.exp(-np.arange(N[0]) / 3.0)[:, None, None]
    V = [1e-3 * damp * (rng.standard_normal(o.cshape) + 1j * rng.standard_normal(o.cshape)) for _ in range(3)]
    for v in V:
        v[:, :, 0] = 0.5 * (v[:, :, 0] + np.conj(v[:, (-np.arange(N[1])) % N[1], 0]))
    b = api.ChFF_Basis(N, kfactor=KF)
    S = dev(V[0])
    B = b.complex_array()
    # the bounds of the other Chebyshev tests: transforms and derivative 1e-13
    # (12 for the nonlinear term), solves and steps 1e-11, pressure 1e-10; the
    # derivative sums and the wall sums of k^2 grow round-off with the length
    grow = max(1.0, (N[0] / 64.0) ** 2)
    b.Xderiv(S, B)
    assert rel_l2(host(B), o.cheb_xderiv(V[0])) <= 1e-13 * grow
    b.Helmholtz(S, B, 3.5, 0.25 + 0.5j, -1.0j)
    assert rel_l2(host(B), o.helmholtz(V[0], 3.5, 0.25 + 0.5j, -1.0j)) <= 1e-11 * grow
    U = api.FluidVF(b, 0.05)
    U.set_field([dev(v) for v in V])
    ta = api.Time_advance_incompress_BDF1(U, 1e-3)
    ta.Compute_nlin()
    assert rel_l2_vec([host(n) for n in U.nlin], o.compute_nlin_chff([v.copy() for v in V])) <= 1e-12 * grow
    ta.Time_advance_step(2)
    for _ in range(2):
        P = o.bdf1_chff(0.05, 1e-3, V)
    ev, ep = rel_l2_vec([host(v) for v in U.cvf], V), rel_l2(host(ta.P), P)
    log(f"  two steps: velocity {ev:.2e} pressure {ep:.2e}")
    assert ev <= 1e-11 * grow and ep <= 1e-10 * grow
    b.close()
