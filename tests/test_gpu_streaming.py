"""Steps, gradients and transfers past 256 MiB of fields, where the passes take
their non-temporal instances with four wavefronts a z block: kernels that thin
grids with the same line lengths do not reach.  Broadband fields, against the
same equations in torch's FP64 transforms."""
import math

import numpy as np
import pytest

from gpu_util import log

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
from tarang_amd import api  # noqa: E402

# the parity bounds of the step tests: FP64 1e-12 (gradients and transfers 1e-11); FP32 transforms 2e-5 (transfers 1e-4)
TOL = {api.PREC_FP64: 1e-12, api.PREC_FP32: 2e-5}
PRECS = [api.PREC_FP64, api.PREC_FP32]


def _err(got, want):
    num = sum(float(torch.linalg.vector_norm(a - b)) ** 2 for a, b in zip(got, want))
    return math.sqrt(num / sum(float(torch.linalg.vector_norm(b)) ** 2 for b in want))


class Fourier:
    """Spectral operators on (Nx, Ny, Nz/2+1) half spectra; walls: sin/cos series along x."""

    def __init__(self, n, dealias, walls=False):
        self.n, self.walls = n, walls
        i = [torch.arange(m, dtype=torch.float64, device="cuda") for m in (n[0], n[1], n[2] // 2 + 1)]
        self.k = [i[0] if walls else torch.where(i[0] <= n[0] // 2, i[0], i[0] - n[0]), torch.where(i[1] <= n[1] // 2, i[1], i[1] - n[1]), i[2]]
        self.k = [a.reshape([-1 if d == e else 1 for e in range(3)]) for d, a in enumerate(self.k)]
        self.k2 = sum(a * a for a in self.k)
        x = self.k[0] > 2 * n[0] // 3 if walls else self.k[0].abs() > n[0] // 3
        y, z = self.k[1].abs() > n[1] // 3, self.k[2] > n[2] // 3
        if dealias == api.DEALIAS_REF_CORNER:
            # the corner is one index narrower at the upper end of each periodic axis
            ix, iy = (a.reshape([-1 if d == e else 1 for e in range(3)]) for d, a in enumerate(i[:2]))
            x = x if walls else (ix > n[0] // 3) & (ix < 2 * n[0] // 3)
            cut = x & (iy > n[1] // 3) & (iy < 2 * n[1] // 3) & z
        else:
            cut = x | y | z
        self.keep = (~cut).double()
        m = torch.arange(n[0], device="cuda")
        ph = math.pi * ((m[:, None] * (2 * m[None, :] + 1)) % (4 * n[0])).double() / (2 * n[0])   # mode, point
        self.series = {False: torch.cos(ph), True: torch.sin(ph)}

    def _x(self, a, m):
        return torch.complex(torch.tensordot(m, a.real, dims=([1], [0])), torch.tensordot(m, a.imag, dims=([1], [0])))

    def inv(self, a, sine=False):
        if self.walls:
            w = torch.full((self.n[0],), 2.0, dtype=torch.float64, device="cuda")
            w[0] = 0.0 if sine else 1.0
            a = torch.fft.ifft(self._x(a, self.series[sine].T * w), dim=1, norm="forward")
        else:
            a = torch.fft.ifft2(a, dim=(0, 1), norm="forward")
        edge = torch.zeros(a.shape[2], dtype=torch.bool, device="cuda")
        edge[0] = edge[-1] = True
        a = torch.complex(a.real, torch.where(edge, 0.0, a.imag))
        return torch.fft.irfft(a, n=self.n[2], dim=2, norm="forward")

    def fwd(self, r, sine=False):
        if not self.walls:
            return torch.fft.fft2(torch.fft.rfft(r, dim=2, norm="forward"), dim=(0, 1), norm="forward")
        a = torch.fft.fft(torch.fft.rfft(r, dim=2, norm="forward"), dim=1, norm="forward")
        return self._x(a, self.series[sine] / self.n[0])

    def div(self, u, w):
        return [1j * sum(self.k[j] * self.fwd(u[j] * w[i]) for j in range(3)) for i in range(3)]

    def solenoidal(self, v):
        p = sum(k * a for k, a in zip(self.k, v)) / self.k2.clamp(min=1.0)
        return [a - k * p for a, k in zip(v, self.k)]

    def noise(self, seed, energy, sine=False):
        """Modes of every wavenumber, conjugate symmetric, none on the Nyquist planes."""
        g = torch.Generator(device="cuda").manual_seed(seed)
        a = self.fwd(torch.randn(self.n, dtype=torch.float64, device="cuda", generator=g), sine) * (1 + self.k2) ** -0.9
        if not self.walls:
            a[self.n[0] // 2] = 0
        a[:, self.n[1] // 2] = 0
        a[:, :, -1] = 0
        return a * math.sqrt(energy / float(torch.linalg.vector_norm(a)) ** 2)

    def flow(self, seed, energy):
        return self.solenoidal([self.noise(seed + c, energy / 3) for c in range(3)])

    def reality(self, a):
        """Conjugate symmetric kz = 0 plane from its first half, empty kz = Nz/2 plane."""
        nx, ny, _ = self.n
        a, p = a.clone(), a[:, :, 0].clone()
        lower = torch.zeros((nx, ny), dtype=torch.bool, device="cuda")
        lower[nx // 2 + 1:] = True
        lower[:, ny // 2] = False
        lower[0, ny // 2 + 1:] = True
        a[:, :, 0] = torch.where(lower, torch.roll(torch.flip(p, (0, 1)), (1, 1), (0, 1)).conj(), p)
        a[:, :, -1] = 0
        return a

    def lawson(self, v0, rates, rhs, dt):
        eh = [torch.exp(-r * self.k2 * 0.5 * dt) for r in rates]
        k = rhs(v0)
        v = [e * (self.keep * a + 0.5 * dt * r) for e, a, r in zip(eh, v0, k)]
        acc = [e * e * r * (dt / 6) for e, r in zip(eh, k)]
        k = rhs(v)
        v = [e * a + 0.5 * dt * r for e, a, r in zip(eh, v0, k)]
        acc = [s + e * r * (dt / 3) for s, e, r in zip(acc, eh, k)]
        k = rhs(v)
        v = [e * (e * a + dt * r) for e, a, r in zip(eh, v0, k)]
        acc = [s + e * r * (dt / 3) for s, e, r in zip(acc, eh, k)]
        return [e * e * a + s + r * (dt / 6) for e, a, s, r in zip(eh, v0, acc, rhs(v))]

    def ns(self, v):
        u = [self.inv(self.keep * a) for a in v]
        return [-a for a in self.solenoidal(self.div(u, u))]


def _velocity(basis, v, nu):
    u = api.FluidVF(basis, nu)
    u.set_field([a.clone() for a in v])
    return u


# the last two: tiles with rows of less than 128 bytes
@pytest.mark.parametrize("dealias", [api.DEALIAS_REF_CORNER, api.DEALIAS_TWOTHIRDS])
@pytest.mark.parametrize("n,prec", [((256, 256, 256), api.PREC_FP64), ((256, 256, 512), api.PREC_FP32), ((1024, 128, 128), api.PREC_FP64),
                                    ((512, 256, 128), api.PREC_FP32)])
def test_ns(n, prec, dealias):
    nu, dt = 5e-3, 1e-3
    f = Fourier(n, dealias)
    v = f.flow(1, 0.5)
    b = api.FFF_Basis(n, precision=prec, dealias=dealias, strong_reality=True)
    u = _velocity(b, v, nu)
    api.Time_advance_incompress(u, dt).Time_advance_step(1)
    e = _err(u.cvf, [f.reality(a) for a in f.lawson(v, [nu] * 3, f.ns, dt)])
    log(f"ns {n} {prec} {dealias}: {e:.3e}")
    assert e <= TOL[prec]
    b.close()


@pytest.mark.parametrize("n,prec", [((256, 128, 256), api.PREC_FP64), ((256, 256, 256), api.PREC_FP32), ((960, 64, 128), api.PREC_FP64),
                                    ((512, 128, 256), api.PREC_FP32)])
def test_mhd(n, prec):
    nu, dt = 5e-3, 1e-3
    f = Fourier(n, api.DEALIAS_TWOTHIRDS)
    v, w = f.flow(1, 0.5), f.flow(11, 0.25)

    def rhs(z):
        u, m = ([f.inv(f.keep * a) for a in z[3 * i:3 * i + 3]] for i in range(2))
        nu_ = f.solenoidal([p - q for p, q in zip(f.div(u, u), f.div(m, m))])
        return [-a for a in nu_] + [q - p for p, q in zip(f.div(u, m), f.div(m, u))]

    b = api.FFF_Basis(n, precision=prec, dealias=api.DEALIAS_TWOTHIRDS, strong_reality=True)
    u, m = _velocity(b, v, nu), _velocity(b, w, nu)
    api.Time_advance_incompress_MHD(u, m, dt).Time_advance_step(1)
    e = _err(u.cvf + m.cvf, [f.reality(a) for a in f.lawson(v + w, [nu] * 6, rhs, dt)])
    log(f"mhd {n} {prec}: {e:.3e}")
    assert e <= TOL[prec]
    b.close()


@pytest.mark.parametrize("prec", PRECS)
def test_rbc(prec):
    n, ra, dt = ((256, 128, 256), (256, 256, 256))[prec], 1e4, 1e-3
    f = Fourier(n, api.DEALIAS_TWOTHIRDS, walls=True)
    sine = (True, False, False, True)
    z = [f.noise(1 + c, 0.01, s) for c, s in enumerate(sine)]
    for c in (0, 3):
        z[c][0] = 0
    dx = lambda a, s: (f.k[0] if s else -f.k[0]) * a

    def rhs(v):
        r = [f.inv(f.keep * a, s) for a, s in zip(v, sine)]
        out = []
        for i in range(4):
            p = [f.fwd(r[j] * r[i], sine[i] != sine[j]) for j in range(3)]
            out.append(dx(p[0], sine[i] != sine[0]) + 1j * (f.k[1] * p[1] + f.k[2] * p[2]))
        out[0], out[3] = out[0] - v[3], out[3] - v[0]
        p = (f.k[0] * out[0] + 1j * (f.k[1] * out[1] + f.k[2] * out[2])) / f.k2.clamp(min=1.0)
        return [f.k[0] * p - out[0], -out[1] - 1j * f.k[1] * p, -out[2] - 1j * f.k[2] * p, -out[3]]

    b = api.SFF_Basis(n, kfactor=(1.0, 1.0, 1.0), precision=prec, dealias=api.DEALIAS_TWOTHIRDS, reality=0)
    u, t = _velocity(b, z[:3], 0.0), api.FluidSF(b)
    t.set_field(z[3].clone())
    api.Time_advance_incompress_RBC(u, t, ra, 1.0, dt).Time_advance_step(1)
    e = _err(u.cvf + [t.F], f.lawson(z, [ra ** -0.5] * 4, rhs, dt))
    log(f"rbc {n} {prec}: {e:.3e}")
    assert e <= TOL[prec]
    b.close()


@pytest.mark.parametrize("prec", PRECS)
def test_gradient(prec):
    """Two steps and the sweep back: every mode of the fused backward pass."""
    n, nu, dt = ((256, 256, 256), (256, 256, 512))[prec], 5e-3, 1e-3
    f = Fourier(n, api.DEALIAS_REF_CORNER)
    v = f.flow(1, 0.5)
    b = api.FFF_Basis(n, precision=prec, dealias=api.DEALIAS_REF_CORNER, strong_reality=False)
    u = _velocity(b, v, nu)
    adj = api.Adjoint_incompress(u, dt)
    adj.Forward(2)
    got = [a.clone() for a in u.cvf]
    adj.Backward(got)                    # of half the sum of squares
    # step by step, so that one step's graph is held at a time
    v1 = f.lawson(v, [nu] * 3, f.ns, dt)
    lam = f.lawson(v1, [nu] * 3, f.ns, dt)
    e_f = _err(u.cvf, lam)
    for at in (v1, v):
        at = [a.detach().clone().requires_grad_(True) for a in at]
        lam = list(torch.autograd.grad(f.lawson(at, [nu] * 3, f.ns, dt), at, [a.detach() for a in lam]))
    e = _err(got, lam)
    log(f"gradient {n} {prec}: forward {e_f:.3e}, backward {e:.3e}")
    assert e_f <= TOL[prec] and e <= (1e-11 if prec == api.PREC_FP64 else 2e-5)
    b.close()


@pytest.mark.parametrize("dealias", [api.DEALIAS_REF_CORNER, api.DEALIAS_TWOTHIRDS])
@pytest.mark.parametrize("prec", PRECS)
def test_transfers(prec, dealias):
    """The giver passes, cut by the 2/3 rule and the giver's radius."""
    n = ((256, 256, 256), (256, 256, 512))[prec]
    f = Fourier(n, dealias)
    v = [f.keep * a for a in f.flow(1, 0.5)]
    radii = np.array([0.0, 4.0, 16.0, 50.0, np.inf])
    b = api.FFF_Basis(n, precision=prec, dealias=dealias)
    flux, s = api.EnergyTr(b, radii, radii).Compute_flux_and_shell_tr(_velocity(b, v, 0.0))
    u, k = [f.inv(a) for a in v], f.k2.sqrt().expand(v[0].shape).contiguous()
    at = torch.searchsorted(torch.from_numpy(radii).to("cuda"), k).reshape(-1)
    mult = torch.where(f.k[2] > 0, 2.0, 1.0).double() * torch.where((f.k[0] == n[0] // 2) | (f.k[1] == n[1] // 2), 2.0, 1.0)
    nr = len(radii)
    S, T = np.zeros((nr, nr)), np.zeros((nr, nr))
    for g in range(1, nr - 1):
        w = [f.inv(((k > radii[g - 1]) & (k <= radii[g])) * a) for a in v]
        d = mult * sum((a * c.conj()).real for a, c in zip(f.div(u, w), v))
        for to, d_ in ((T, d), (S, d * (k <= min(n) // 2))):
            to[g] = [-float(d_.reshape(-1)[at == i].sum()) for i in range(nr)]
    F = np.array([0.0] + [T[1:i + 1, i + 1:].sum() for i in range(1, nr)])
    e = [np.linalg.norm(a - c) / np.linalg.norm(c) for a, c in ((s, S), (flux, F))]
    log(f"transfers {n} {prec} {dealias}: shells {e[0]:.3e}, flux {e[1]:.3e}")
    assert max(e) <= (1e-11 if prec == api.PREC_FP64 else 1e-4)
    b.close()
