"""Layers on clumped absolute positions, enough of them that the sort keeps
lists, on a mesh of 512 large tiles: the forward's sort handed to the
backward's three-component paint against a sort of its own, and lists in the
spectra's room against none.  The paints add integers, so every output keeps
its bits."""
import numpy as np
import pytest
import torch

from jerald_amd import _lib as L
from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh

pytestmark = pytest.mark.gpu

SIDE, NM = 162, (128, 128, 128)  # 162^3 > 2^22 particles


def model(dtype, **kw):
    rng = np.random.default_rng(3)
    n = SIDE**3
    i = np.arange(n)
    X = np.stack((i // SIDE**2, i // SIDE % SIDE, i % SIDE), -1) * (NM[0] / SIDE) + rng.standard_normal((n, 3))
    m = rng.random(n) < 0.4
    X[m] = (rng.random((200, 3)) * NM)[rng.integers(0, 200, m.sum())] + 1.5 * rng.standard_normal((m.sum(), 3))
    pm = PMesh(NM, tuple(float(v) for v in NM), dtype=dtype)
    return JERALDModel(torch.tensor(np.mod(X, NM)), torch.tensor(rng.random(NM)), pm, Nstep=1, kind="dm", **kw)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_outputs_for_every_way_to_sort(dtype):
    p = torch.tensor([0.2, 0.7, 0.9, 4.0, 0.3], dtype=torch.float64)
    want = model(dtype).loss_and_grad_positions(p)
    own = model(dtype, reuse_sort=False).loss_and_grad_positions(p)
    m = model(dtype)
    L.workspaces.clear()
    need = m._ws().numel()
    m._ws_flags = lambda: m.paint_flags | L.LDL_PAINT_LATTICE  # no room for lists
    L.workspaces.clear()
    assert m._ws().numel() < need
    bare = m.loss_and_grad_positions(p)
    for other in (own, bare):
        for a, b in zip(want, other):
            assert torch.equal(a, b)
