"""Absolute positions outside the box, at its faces and on cell faces, through
every decode of the paint's kernels and of the gathers: the paint bitwise
against the CPU emulation (which wraps with the C library's fmod and divides),
the readout against the oracle at the same mesh coordinates."""
import numpy as np
import pytest
import torch

from jerald_amd import jaxpops as J
from oracle import native as NV

pytestmark = pytest.mark.gpu


def positions(box, nm, dt, rng):
    n = 3000
    L, N = np.array(box), np.array(nm)
    x = rng.random((n, 3)) * L
    k = rng.integers(0, 12, (n, 3))
    cell = L / N
    x = np.where(k == 1, x - L, x)                       # one period below
    x = np.where(k == 2, x + L, x)                       # and above
    x = np.where(k == 3, x * 1e6, x)                     # many periods
    x = np.where(k == 4, -x * 37.0, x)
    x = np.where(k == 5, rng.integers(-4, 5, (n, 3)) * L, x)          # whole periods
    x = np.where(k == 6, rng.integers(0, 64, (n, 3)) * cell, x)       # cell faces
    x = np.where(k == 7, -1e-20, x)                      # wraps to the box size itself
    x = np.where(k == 8, 1e-30, x)
    x = x.astype(dt)
    x = np.where(k == 9, np.nextafter(L.astype(dt), dt(0)), x)
    return np.ascontiguousarray(x.astype(dt))


@pytest.mark.parametrize("nm", [(16, 32, 8), (20, 13, 30), (5, 64, 2)], ids=str)
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_absolute_positions_anywhere(nm, dt):
    rng = np.random.default_rng(sum(nm))
    box = (51.3, 20.0, 409.6)
    x = positions(box, nm, dt, rng)
    acc, s = NV.paint_fixed(x, 1.0, nm, box=box, dtype=dt)
    xt = torch.tensor(x, device="cuda")
    got = J.ppaint(xt, 1.0, nm, box).cpu().numpy()
    assert np.array_equal(got, NV.fixed_to_float(acc, s, dt))
    # mesh coordinates in the working precision, as the kernels form them
    L = np.array(box).astype(dt)
    u = np.fmod(x, L)
    u = np.where(u < 0, u + L, u) / (L / np.array(nm).astype(dt))
    field = rng.standard_normal(nm)
    want = NV.readout_f64(u.astype(np.float64) % np.array(nm), field)
    out = J.preadout(xt, torch.tensor(field, device="cuda", dtype=xt.dtype), nm, box).double().cpu().numpy()
    assert np.abs(out - want).max() <= 64 * np.finfo(dt).eps * np.abs(field).max()
