"""The paint's particle sort with and without stray lists: particles in
lattice order, partly and wholly out of order, all in one cell, ragged
numbers around the chunk size and the line where the lists begin.  The
fixed-point paint has to give the same bits for any order and any sort, so
every case is compared with the CPU emulation of it."""
import numpy as np
import pytest
import torch

from jerald_amd import jaxpops as J
from oracle import native as NV

pytestmark = pytest.mark.gpu

KSTRAY = 1 << 22  # particles from which the lists are used


def positions(kind, n, nm, rng):
    side = int(np.ceil(n ** (1 / 3)))
    i = np.arange(n)
    q = np.stack((i // (side * side), (i // side) % side, i % side), -1) * (np.array(nm) / side)
    x = np.mod(q + rng.standard_normal((n, 3)), nm)
    if kind == "clumped":
        m = rng.random(n) < 0.4
        c = rng.random((200, 3)) * nm
        x[m] = np.mod(c[rng.integers(0, 200, m.sum())] + 1.5 * rng.standard_normal((m.sum(), 3)), nm)
    elif kind == "shuffled":
        x = x[rng.permutation(n)]
    elif kind == "one cell":
        x[:] = np.array(nm) / 2 + 0.25
    return x.astype(np.float32)


CASES = [("ordered", KSTRAY + 1, (128, 128, 128)), ("clumped", KSTRAY + 2047, (160, 96, 250)), ("shuffled", KSTRAY, (256, 64, 512)),
         ("one cell", KSTRAY + 77, (64, 64, 64)), ("clumped", KSTRAY - 1, (128, 128, 128)), ("shuffled", 2049, (40, 50, 60)),
         ("clumped", 2048, (16, 16, 16)), ("shuffled", 1, (8, 8, 8)), ("shuffled", KSTRAY, (8, 16, 32))]


@pytest.mark.parametrize("kind,n,nm", CASES, ids=lambda v: str(v))
def test_paint_bits_for_any_order(kind, n, nm):
    rng = np.random.default_rng(n)
    x = positions(kind, n, nm, rng)
    box = tuple(float(v) for v in nm)
    got = J.ppaint(torch.tensor(x, device="cuda"), 1.0, nm, box).cpu().numpy()
    acc, s = NV.paint_fixed(x, 1.0, nm, box=box)
    assert np.array_equal(got, NV.fixed_to_float(acc, s, np.float32))


def test_three_component_paint_for_clumped_particles():
    n, nm = KSTRAY + 3, (96, 100, 128)
    rng = np.random.default_rng(5)
    x = positions("clumped", n, nm, rng)
    m = rng.standard_normal((n, 3)).astype(np.float32)
    box = tuple(float(v) for v in nm)
    got = J.ppaint3D(torch.tensor(x, device="cuda"), torch.tensor(m, device="cuda"), nm, box).cpu().numpy()
    for c in range(3):
        acc, s = NV.paint_fixed(x, m[:, c], nm, box=box)
        assert np.array_equal(got[c], NV.fixed_to_float(acc, s, np.float32))
