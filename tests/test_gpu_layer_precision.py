"""Rounding of the FP64 layer on meshes with factors 3 and 5.  The derivative
symbol multiplies a spectrum, so the forces carry the rounding of the
transforms alone: against the same route in extended precision, from the
layer's own density, they may be off by twice what numpy's FP64 transforms are
(the same operations in another order).  Differences of a rounded potential
are off by 2 to 13 times that under a filter of long waves."""
import numpy as np
import pytest
import torch

from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh

pytestmark = pytest.mark.gpu

CELL = 0.8
PRM = [0.01, 1.0, 0.1, 1.0, 0.0]  # alpha, gamma, kh, kl, nu


def axis(n, half):
    m = np.fft.fftfreq(n, 1.0 / n)
    if half:
        m = m[: n // 2 + 1].copy()
    t = 2 * np.arctan2(np.longdouble(0), np.longdouble(-1)) * m.astype(np.longdouble) / n
    D = (45 * np.sin(t) - 9 * np.sin(2 * t) + np.sin(3 * t)) / (30 * np.longdouble(CELL))
    D[2 * np.abs(m) == n] = 0
    return t / np.longdouble(CELL), D


@pytest.mark.parametrize("nm", [(40, 40, 40), (100, 100, 100), (64, 60, 54), (96, 20, 128)], ids=str)
def test_fp64_forces_carry_the_transforms_rounding_only(nm):
    rng = np.random.default_rng(5)
    box = tuple(CELL * n for n in nm)
    q = np.stack(np.meshgrid(*[np.arange(n) for n in nm], indexing="ij"), -1).reshape(-1, 3)
    wave = [2 * np.pi * q[:, d] / nm[d] for d in range(3)]  # a few long waves, as a density field has
    X = q + 2.0 * np.stack([np.sin(wave[d] + 0.3) + 0.5 * np.cos(2 * wave[(d + 1) % 3]) for d in range(3)], -1)
    X += 0.1 * rng.standard_normal(X.shape)
    m = JERALDModel(torch.tensor(np.mod(X * CELL, box)), torch.zeros(nm), PMesh(nm, box, dtype=torch.float64), Nstep=1, kind="sm")
    _, rho, _, F, _, _ = m._layer_fwd(m.X, PRM, 1.0)
    (kx, Dx), (ky, Dy), (kz, Dz) = (axis(n, d == 2) for d, n in enumerate(nm))
    k2 = kx[:, None, None] ** 2 + ky[None, :, None] ** 2 + kz[None, None, :] ** 2
    k2[0, 0, 0] = np.longdouble(1e-8) ** 2
    a, _, kh, kl, _ = (np.longdouble(v) for v in PRM)
    H = np.longdouble(1e-2) * a * -np.exp(-k2 / kl**2 - kh**2 / k2)
    symbols = (Dx[:, None, None], Dy[None, :, None], Dz[None, None, :])

    def forces(T):  # gamma = 1; the forward's 1 / N^3 and the inverse's cancel
        P = H.astype(T) * np.fft.rfftn(rho.cpu().numpy().astype(T) + T(1e-8))
        assert P.real.dtype == T
        return [np.fft.irfftn(-1j * D.astype(T) * P, s=nm, axes=(0, 1, 2)) for D in symbols]

    F = F.cpu().numpy()
    for d, (want, f64) in enumerate(zip(forces(np.longdouble), forces(np.float64))):
        err, err64 = (np.sqrt(np.mean((f - want) ** 2)) for f in (F[..., d], f64))
        assert err <= 2 * err64, (d, float(err / err64))
