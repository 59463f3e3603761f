"""The real-space derivative stencils of the layer on every route of their
dispatch: the direct kernels (up to 2^20 cells), the marching ones at each
tile width, partial tiles and partial chunks, and meshes thinner than the
stencil.  Loss and every gradient, positions included, against the FP64
oracle: FP64 with the tolerances of the model's own parity tests; FP32, on
densities this sparse (up to 512 mean densities a particle), within 1e-3 of
the gradients' norms, which a wrong neighbour misses by orders."""
import numpy as np
import pytest
import torch

from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh
from oracle import ldl_oracle as O

pytestmark = pytest.mark.gpu

MESHES = [
    (4, 8, 8),         # direct, x axis shorter than the stencil's reach
    (64, 16, 1024),    # direct, exactly 2^20 cells
    (32, 64, 1024),    # march, 64 cells wide, 4-plane chunks
    (1024, 8, 256),    # march, y tile half empty
    (64, 256, 1024),   # march, 2^24 cells: widest tiles
    (1024, 128, 128),  # march, 2^24 cells: 128 wide in both precisions
]


@pytest.mark.parametrize("nm", MESHES, ids=str)
@pytest.mark.parametrize("dt", [torch.float64, torch.float32], ids=["f64", "f32"])
def test_layer_with_stencils_matches_oracle(nm, dt):
    rng = np.random.default_rng(91)
    cell = 0.8
    box = np.array(nm) * cell
    lat = tuple(min(n, 32) for n in nm)
    q = np.stack(np.meshgrid(*[np.arange(l) * (b / l) for l, b in zip(lat, box)], indexing="ij"), -1).reshape(-1, 3)
    X = q + cell * rng.standard_normal(q.shape)
    tgt = 0.5 * rng.random(nm)
    p = np.array([.1, .5, 1., 8., 0.1, 1.1, 0.9, 0.05])
    orc = O.SMModelOracle(nm, box, 1, tgt, L1=False, backend="native")
    loss0, g0, gx0 = orc.loss_and_grad(p, X, want_pos_grad=True)
    m = JERALDModel(torch.tensor(X), tgt, PMesh(nm, box, device="cuda", dtype=dt), Nstep=1, kind="sm", L1=False, lattice=lat)
    loss, g, gx = m.loss_and_grad_positions(torch.tensor(p))
    lt, gt = (1e-10, 1e-8) if dt == torch.float64 else (1e-4, 1e-3)
    assert abs(loss.item() / loss0 - 1) <= lt
    for got, want in ((g, g0), (gx, gx0)):
        d = got.double().cpu().numpy() - want
        assert np.linalg.norm(d) <= gt * np.linalg.norm(want)
