"""Transform lengths with factors 3 and 5, one axis at a time: every kind of
stage group (single radices, the fused pairs, four-group plans), one to many
tiles with ragged last ones, both pencil counts.  Against numpy, with the
tolerances of the other transform tests."""
import numpy as np
import pytest
import torch

from jerald_amd import jaxpops as J
from oracle import ldl_oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [5, 6, 9, 10, 12, 15, 30, 36, 45, 100, 162, 192, 250, 375, 384, 500, 512 + 128, 625, 675, 729, 750, 810, 864, 900, 960, 972, 1000]


def shapes(n):
    out = [(n, 3 * 5, 36), (5, n, 22 + 2)]
    if n % 2 == 0:
        out.append((5, 9, n))
    return out


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("dt", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_axis_of_any_length_matches_numpy(n, dt):
    rng = np.random.default_rng(n)
    rt = 3e-6 if dt == torch.float32 else 1e-13
    for shape in shapes(n):
        x = rng.standard_normal(shape)
        X = np.fft.rfftn(x)
        got = J.pfft(torch.tensor(x, device="cuda", dtype=dt)).cpu().numpy()
        assert np.abs(got - X).max() <= rt * np.abs(X).max() * np.log2(x.size), shape
        Y = rng.standard_normal(X.shape) + 1j * rng.standard_normal(X.shape)
        want = O.pifft(Y, shape)
        got = J.pifft(torch.tensor(Y, device="cuda", dtype=torch.complex64 if dt == torch.float32 else torch.complex128), shape)
        assert np.abs(got.cpu().numpy() - want).max() <= rt * np.abs(want).max() * np.log2(x.size), shape
