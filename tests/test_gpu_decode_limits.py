"""The position decode at the limits of its inputs: a box that rounds to zero
in the working precision, lattice points beyond 32-bit cell numbers."""
import numpy as np
import pytest
import torch

from jerald_amd import _lib as L
from jerald_amd import jaxpops as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm", [(8, 16, 4), (6, 10, 15)], ids=str)
def test_box_that_rounds_to_zero_reads_nan(nm):
    x = torch.tensor([[0.0, 0.0, 0.0], [1.5, -2.0, 1e-30], [-1e30, 3e38, 1e-45]], device="cuda")
    out = J.preadout(x, torch.ones(nm, device="cuda"), nm, (1e-46,) * 3)
    assert np.isnan(out.cpu().numpy()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("step", [1e6 + 0.25, 2.0**31, 2.0**32 - 6, 1e10, 3e14 + 1])
def test_lattice_points_far_from_the_first(step, dtype):
    nm, lat = (20, 13, 30), (5, 4, 3)
    n = int(np.prod(lat))
    rng = np.random.default_rng(2)
    step = np.array([step, 2.5, step + 1])
    i = np.stack(np.meshgrid(*[np.arange(m) for m in lat], indexing="ij"), -1).reshape(-1, 3)
    move = rng.integers(-3, 4, (n, 3))
    d = move - (i * step) % 1  # every particle on a cell: it reads that cell's value
    cell = (np.floor(i * step) + move).astype(np.int64)
    idx = [cell[:, a] % nm[a] for a in range(3)]
    field = rng.standard_normal(nm)
    x = torch.tensor(d, dtype=dtype, device="cuda")
    f = torch.tensor(field, dtype=dtype, device="cuda")
    out, rho = torch.empty(n, dtype=dtype, device="cuda"), torch.empty(nm, dtype=dtype, device="cuda")
    pd = L.pos_desc(tuple(float(v) for v in nm), L.LDL_POS_LATTICE, lat, step)
    L.call(f"ldl_preadout_{L.sfx(dtype)}", L.ptr(x), pd, n, L.ptr(f), L.i64x3(nm), -1, L.ptr(out), L.stream_ptr(x.device))
    assert torch.equal(out, f[tuple(torch.tensor(v, device="cuda") for v in idx)])
    nb = L.load().ldl_paint_workspace_bytes(L.i64x3(nm), 1, n, 0)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    L.call(f"ldl_ppaint_{L.sfx(dtype)}", L.ptr(x), pd, n, None, 1.0, L.i64x3(nm), 1.0, 0, L.ptr(rho), L.ptr(ws), nb, L.stream_ptr(x.device))
    want = np.zeros(nm)
    np.add.at(want, tuple(idx), 1.0)
    assert np.array_equal(rho.double().cpu().numpy(), want)


def test_subnormal_cells_wrap_as_the_division_rounds():
    # L / N rounds by up to a part in a few: coordinates run past N and wrap
    nm, L = (5, 6, 1000), np.float32(1e-41)
    box = (float(L),) * 3
    rng = np.random.default_rng(4)
    x = (rng.random((500, 3)) * float(L) * 0.999).astype(np.float32)
    u = x / (L / np.array(nm, dtype=np.float32))
    assert u.dtype == np.float32 and (u[:, 2] > 1001).any()
    i = np.floor(u).astype(int)
    field = rng.standard_normal(nm).astype(np.float32)
    want = np.zeros(500)
    for a in range(8):
        b = np.array([a >> 2, a >> 1, a]) & 1
        w = np.prod(np.where(b, u - i, 1 - (u - i)).astype(float), axis=1)
        want += w * field[tuple(((i + b) % nm).T)]
    out = J.preadout(torch.tensor(x, device="cuda"), torch.tensor(field, device="cuda"), nm, box).double().cpu().numpy()
    assert np.abs(out - want).max() <= 8 * np.finfo(np.float32).eps * np.abs(field).max()
