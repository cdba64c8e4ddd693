"""The line lengths of the wavefront x pass (second half of its list) and of
the two-step pencil passes beyond 160 points, with a full spectrum: step,
max Σ|v| and transforms against the same scheme in FP64 ``torch.fft``."""
import numpy as np
import pytest
import torch

import distributednavierstokes_amd as dns
from distributednavierstokes_amd.spectral import DeviceState

pytestmark = pytest.mark.gpu

VISC = 1e-3
WRAY = ((8 / 15, 1 / 4, 8 / 15), (5 / 12, 0.0, 2 / 15), (3 / 4, 0.0, 1 / 3))  # a, b of Δt du; share of Δt of the viscous factor


class Torch:
    """States are (c, kz, ky, kx) on the retained modes, kz and ky wrapped."""

    def __init__(self, n, kcut):
        self.n, self.kcut = n, kcut
        dev = "cuda"
        k = torch.cat([torch.arange(kcut + 1, device=dev), torch.arange(-kcut, 0, device=dev)])
        self.idx = k % n
        k = k.double()
        self.k = (torch.arange(kcut + 1, device=dev).double()[None, None, :], k[None, :, None], k[:, None, None])
        self.k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2

    def cut(self, a):
        return torch.fft.rfftn(a, norm="forward")[self.idx][:, self.idx][:, :, : self.kcut + 1]

    def physical(self, uh):
        out = []
        for a in uh:
            f = torch.zeros((self.n, self.n, self.n // 2 + 1), dtype=torch.complex128, device="cuda")
            f[self.idx[:, None, None], self.idx[None, :, None], torch.arange(self.kcut + 1, device="cuda")[None, None]] = a
            out.append(torch.fft.irfftn(f, s=(self.n,) * 3, norm="forward"))
        return out

    def project(self, uh):
        div = sum(k * a for k, a in zip(self.k, uh)) / self.k2.clamp(min=1)
        return torch.stack([a - k * div for k, a in zip(self.k, uh)])

    def field(self, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        uh = torch.stack([self.cut(torch.randn((self.n,) * 3, generator=g, device="cuda", dtype=torch.float64))
                          for _ in range(3)])
        uh[:, 0, 0, 0] = 0
        uh = self.project(uh)
        return uh / (2 * uh.abs().square().sum()).sqrt()

    def rhs(self, uh):
        v = self.physical(uh)
        du = torch.zeros_like(uh)
        for i in range(3):
            for j in range(i, 3):
                s = self.cut(v[i] * v[j])
                du[i] -= 1j * self.k[j] * s
                if i != j:
                    du[j] -= 1j * self.k[i] * s
        return du, float((v[0].abs() + v[1].abs() + v[2].abs()).max())

    def step(self, uh, dt):
        start, vmax = uh, None
        for a, b, c in WRAY:
            du, vm = self.rhs(uh)
            vmax = vm if vmax is None else vmax
            phi = torch.exp(-VISC * c * dt * self.k2)
            uh, start = self.project(phi * (start + a * dt * du)), phi * (start + b * dt * du)
        return uh, vmax


def host(uh):
    """(kx, ky, kz, c) column-major, as the library takes it."""
    return uh.cpu().numpy().transpose(3, 2, 1, 0)


def device(a):
    return torch.as_tensor(np.ascontiguousarray(a.transpose(3, 2, 1, 0)), device="cuda")


# x lines: n = 2·12·8 ... 2·16·16, FP64 up to N2 = 12 (the others by the block kernels); pencils: every even
# length of the lists from 162 on; the IF stage by either kernel; 64-row slabs in FP32 from 256 on, the last one
# ragged at 270 ... 360; kcut at n / 3 and well below it
FP32 = [162, 180, 192, 200, 216, 240, 250, 256, 270, 288, 300, 320, 324, 360, 384, 400, 432, 450, 480, 486, 500]
FP64 = [180, 192, 200, 240, 256, 270, 288, 300, 320, 384, 432]


@pytest.mark.parametrize("n,kcut,T", [(n, n // 3, np.float32) for n in FP32] + [(n, n // 3, np.float64) for n in FP64]
                         + [(n, 40, T) for n in (240, 384) for T in (np.float32, np.float64)])
def test_step_and_transforms(n, kcut, T):
    """1e-12 (FP64) and 2e-5 (FP32) of the field's maximum, the bounds of the
    shorter lines' tests.  All modes of the field are equally strong and Δt is
    half the inverse cutoff, so a mode that a pass loses, or a wrong increment
    of one, shows at the size of the field."""
    tol = 1e-12 if T == np.float64 else 2e-5
    ref = Torch(n, kcut)
    uh, dt = ref.field(n), 0.5 / kcut
    s = dns.spectral_setup(n=n, visc=VISC, kcut=kcut, T=T)
    s.upload(host(uh))
    vm = dns.spectral_step_(DeviceState(s), s, dt)
    want, vr = ref.step(uh, dt)
    got = device(s.download())
    err = float((got - want).abs().max() / want.abs().max())
    print(f"n={n} kcut={kcut} {T.__name__}: step {err:.2e} vmax {abs(vm - vr) / vr:.2e}", flush=True)
    assert abs(vm - vr) <= tol * vr
    assert err <= tol
    if n > 324:
        return
    v = torch.stack(ref.physical(uh))
    vg = np.zeros((n, n, n, 3), order="F")
    dns.spec_to_phys_(vg, host(uh), s)
    assert float((device(vg) - v).abs().max()) <= tol * float(v.abs().max())
    w = np.zeros(s.state_shape, dtype=np.complex128, order="F")
    dns.phys_to_spec_(w, host(v), s)
    assert float((device(w) - uh).abs().max()) <= tol * float(uh.abs().max())


def test_step_beyond_the_tables():
    """n = 540 FP32: the lines that no two-step pass serves."""
    test_step_and_transforms(540, 180, np.float32)
