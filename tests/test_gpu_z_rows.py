"""The z passes on whole padded rows: the longest and the ragged line lengths,
and fields past 256 MiB, where loads and stores bypass the caches."""
import numpy as np
import pytest

from gpu_util import log

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

# FP64 1e-12 and FP32 transforms 2e-5, the parity bounds of the step tests
TOL = {api.PREC_FP64: 1e-12, api.PREC_FP32: 2e-5}


@pytest.mark.parametrize("N", [(8, 8, 16), (8, 16, 48), (16, 8, 240), (8, 8, 640), (8, 8, 1024), (64, 512, 1024)])
def test_transforms(N):
    g = torch.Generator(device="cuda").manual_seed(5)
    b = api.FFF_Basis(N)
    x = torch.randn(N, dtype=torch.float64, device="cuda", generator=g)
    want = (torch.fft.rfftn(x) / x.numel()).contiguous()
    A = torch.full_like(want, float("nan"))
    # rows of nz + 2, the last two not part of the field
    xp = torch.nn.functional.pad(x, (0, 2))
    y = torch.full_like(xp, float("nan"))
    b.Forward_transform(xp, A)
    b.Inverse_transform(want, y)
    y = y[..., :-2]
    e_f = float((A - want).norm() / want.norm())
    e_i = float((y - x).norm() / x.norm())
    log(f"{N}: forward {e_f:.3e}, inverse {e_i:.3e}")
    assert max(e_f, e_i) <= 1e-12
    b.close()


@pytest.mark.parametrize("N,prec", [((8, 8, 48), api.PREC_FP64), ((16, 8, 16), api.PREC_FP32), ((64, 512, 1024), api.PREC_FP64),
                                    ((128, 512, 1024), api.PREC_FP32)])
def test_beltrami_decay(N, prec):
    """A Beltrami wave is its own curl, so its products leave no force: it
    decays as exp(-nu k^2 t), whatever the grid."""
    nu, dt, steps, k = 0.1, 1e-3, 2, 2
    V = [torch.zeros((N[0], N[1], N[2] // 2 + 1), dtype=torch.complex128, device="cuda") for _ in range(3)]
    a, b, c = 1.0, 0.7, 0.4
    # u = a sin kz + c cos ky, v = b sin kx + a cos kz, w = c sin ky + b cos kx
    V[0][0, 0, k] += -0.5j * a
    V[1][0, 0, k] += 0.5 * a
    for s in (1, -1):
        V[0][0, s * k, 0] += 0.5 * c
        V[2][0, s * k, 0] += -0.5j * s * c
        V[1][s * k, 0, 0] += -0.5j * s * b
        V[2][s * k, 0, 0] += 0.5 * b
    want = [v * np.exp(-nu * k * k * dt * steps) for v in V]
    basis = api.FFF_Basis(N, precision=prec)
    U = api.FluidVF(basis, nu)
    U.set_field([v.clone() for v in V])
    api.Time_advance_incompress(U, dt).Time_advance_step(steps)
    err = sum(float((g - w).norm()) ** 2 for g, w in zip(U.cvf, want)) ** 0.5 / sum(float(w.norm()) ** 2 for w in want) ** 0.5
    log(f"{N} {prec}: {err:.3e}")
    assert err <= TOL[prec]
    basis.close()
