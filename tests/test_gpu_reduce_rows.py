"""Shell-binned reductions at the row lengths where a wavefront's 64 modes of a
row end: rows of one wavefront or less, one and two modes more, several
wavefronts with a remainder, fewer rows than blocks and non-cubic boxes
(kfactor), against numpy sums of the same modes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402


def _modes(b):
    k = [np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n) for n in (b.Nx, b.Ny)] + [np.arange(b.Nz // 2 + 1)]
    K = [k[d].reshape([-1 if i == d else 1 for i in range(3)]) * b.kfactor[d] for d in range(3)]
    m = np.where(k[2] > 0, 1.0, 0.5).reshape(1, 1, -1) * np.where((k[0].reshape(-1, 1, 1) == b.Nx // 2) |
                                                                  (k[1].reshape(1, -1, 1) == b.Ny // 2), 2.0, 1.0)
    return np.sqrt(K[0] ** 2 + K[1] ** 2 + K[2] ** 2), m * np.ones(b.shape_complex_array)


@pytest.mark.parametrize("N,kf", [((8, 8, 16), (1.0, 1.0, 1.0)), ((16, 8, 128), (1.0, 2.0, 0.5)), ((8, 24, 256), (1.0, 1.0, 1.0)),
                                  ((40, 16, 96), (0.5, 1.0, 1.5)), ((8, 8, 1024), (1.0, 1.0, 1.0))])
def test_spectrum_and_shells(N, kf):
    b = api.FFF_Basis(N, kfactor=kf, dealias=api.DEALIAS_NONE, strong_reality=True)
    rng = np.random.default_rng(11)
    U = api.FluidVF(b)
    V = [rng.standard_normal(b.shape_complex_array) + 1j * rng.standard_normal(b.shape_complex_array) for _ in range(3)]
    U.set_field(V)
    K, m = _modes(b)
    top = b.Min_radius_outside()
    idx = np.ceil(K).astype(int).ravel()
    val = (m * np.abs(V[0]) ** 2 * K * K).ravel()
    cnt = np.bincount(idx, (2 * m).ravel(), minlength=top + 1)[:top + 1]
    ref = np.bincount(idx, val, minlength=top + 1)[:top + 1] * 4 * np.pi / np.where(cnt > 0, cnt, 1) / np.prod(kf)
    got = b.Compute_shell_spectrum(U.V1)
    # sums of at most 1e5 terms of one sign: n eps / 2 in the reference's own order
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
    # the two binnings of the transfer against each other: the flux summed from the binning without the cut, the
    # matrix from the one inside the largest inscribed sphere
    r = np.array([0.0, 1.5, 3.0, float(b.Max_radius_inside()), np.inf])
    et = api.EnergyTr(b, flux_radii=r, shell_radii=r)
    flux, S = et.Compute_flux_and_shell_tr(U)
    f2, S2 = et.Compute_flux(U), et.Compute_shell_tr(U)
    scale = np.abs(S2).max() + np.abs(f2).max()
    assert np.abs(S - S2).max() <= 1e-12 * scale
    assert np.abs(flux - f2).max() <= 1e-11 * scale
