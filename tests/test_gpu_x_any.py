"""The fused x pass of layers whose x length has factors 3 and 5, at lengths on
both sides of its launch shapes (pencils, threads), with column counts that
leave partial strips: the FP64 model's loss and gradient against the oracle,
the FP32 spectrum against numpy's transform of the FP32 density."""
import numpy as np
import pytest
import torch

from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh
from oracle import ldl_oracle as O

pytestmark = pytest.mark.gpu

MESHES = [(5, 8, 6), (6, 4, 10), (45, 20, 30), (100, 12, 18), (243, 6, 10), (540, 5, 8), (810, 6, 8), (960, 4, 12), (1000, 5, 6), (12, 96, 180)]


@pytest.mark.parametrize("kind", ["sm", "dm", "HI"])
@pytest.mark.parametrize("nm", MESHES, ids=str)
def test_fused_x_pass(nm, kind):
    rng = np.random.default_rng(11)
    box = tuple(float(n) for n in nm)
    q = np.stack(np.meshgrid(*[np.arange(n) for n in nm], indexing="ij"), -1).reshape(-1, 3)
    X = np.mod(q + 0.6 * rng.standard_normal(q.shape), nm)
    star = rng.random(nm) + 0.1
    target = rng.random(nm)
    layer = [0.2, 0.7, 0.9, 4.0, 0.3] + ([0.1, 0.8, 1.1, 3.0, 0.2] if kind == "HI" else [])
    resp = {"sm": [0.9, 1.1, 0.05], "dm": [], "HI": [0.9, 1.1, 0.05, 0.3, 0.9, 4.0, 0.2, 0.3, 0.8, 1.1, 0.05, 0.1]}[kind]
    p = np.array(layer + resp)
    L1 = kind != "dm"
    loss0, g0 = O.SMModelOracle(nm, box, 1, target, L1=L1, kind=kind, starmap=star).loss_and_grad(p, X)
    m = JERALDModel(torch.tensor(X), torch.tensor(target), PMesh(nm, box, dtype=torch.float64), Nstep=1, kind=kind, L1=L1, starmap=torch.tensor(star))
    loss, grad = m.loss_and_grad(torch.tensor(p))
    assert abs(loss.item() - loss0) <= 1e-10 * abs(loss0)
    np.testing.assert_allclose(grad.cpu().numpy(), g0, rtol=1e-8, atol=1e-12 * np.abs(g0).max())
    m = JERALDModel(torch.tensor(X), torch.tensor(target), PMesh(nm, box, dtype=torch.float32), Nstep=1, kind=kind, L1=L1, starmap=torch.tensor(star))
    _, rho, U, _, _, _ = m._layer_fwd(m.X, layer, 1.0)
    want = np.fft.rfftn((rho.double().cpu().numpy() + 1e-8) ** layer[1]) / np.prod(nm)
    got = torch.view_as_complex(U).cpu().numpy()[:, :, : nm[2] // 2 + 1]
    # FP32 power (a few ulp) and transform round-off of the largest bin
    assert np.abs(got - want).max() <= 32 * np.finfo(np.float32).eps * np.abs(want).max()
