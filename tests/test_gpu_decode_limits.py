"""The position decode at the limits of its inputs: a box that rounds to zero
in the working precision."""
import numpy as np
import pytest
import torch

from jerald_amd import jaxpops as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm", [(8, 16, 4), (6, 10, 15)], ids=str)
def test_box_that_rounds_to_zero_reads_nan(nm):
    x = torch.tensor([[0.0, 0.0, 0.0], [1.5, -2.0, 1e-30], [-1e30, 3e38, 1e-45]], device="cuda")
    out = J.preadout(x, torch.ones(nm, device="cuda"), nm, (1e-46,) * 3)
    assert np.isnan(out.cpu().numpy()).all()
