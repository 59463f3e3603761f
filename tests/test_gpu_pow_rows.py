"""The FP64 layer's gamma power over densities from empty cells to dense ones,
through the one-layer density spectrum (rho + 1e-8)^gamma.  Every particle in
one corner leaves many cells at 1e-8; gammas near 0, 1 and 2, a negative one
and one beyond the split exponential's range take every branch (alpha = 0: the
particles stay)."""
import numpy as np
import pytest
import torch

from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh

pytestmark = pytest.mark.gpu

N = 16


@pytest.mark.parametrize("gamma", [-0.5, 0.0, 1e-3, 0.73, 1.0, 2.0, 45.0])
def test_layer_spectrum_power(gamma):
    rng = np.random.default_rng(7)
    X = np.mod(np.concatenate([0.3 * rng.standard_normal((3000, 3)), N * rng.random((500, 3))]), N)
    pm = PMesh(N, float(N), dtype=torch.float64)
    m = JERALDModel(torch.tensor(X), torch.zeros(N, N, N), pm, Nstep=1, kind="dm")
    prm = [0.0, gamma, 0.3, 1.7, 0.4]
    fact = N**3 / X.shape[0]
    _, rho, U, _, _, _ = m._layer_fwd(m.X, prm, fact)
    want = np.fft.rfftn((rho.cpu().numpy() + 1e-8) ** gamma) / N**3
    got = torch.view_as_complex(U).cpu().numpy()[:, :, : N // 2 + 1]
    # transform round-off: a few eps of the largest bin times log2 N per axis
    assert np.abs(got - want).max() <= 64 * np.finfo(float).eps * np.abs(want).max()
