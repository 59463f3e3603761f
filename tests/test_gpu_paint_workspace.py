"""Paints of small meshes in a workspace that has room for the keys of
8 x 16 x 32-cell tiles alone: same bits as in the queried one."""
import numpy as np
import pytest
import torch

from jerald_amd import _lib as L
from jerald_amd import jaxpops as J

pytestmark = pytest.mark.gpu


def large_tile_bytes(nm, n):
    keys = 8 * -(-nm[0] // 8) * -(-nm[1] // 16) * -(-nm[2] // 32)
    al = lambda b: (b + 255) // 256 * 256
    return 256 + 2 * al(4 * (keys + 1)) + al(4 * (keys // 8192 + 1)) + 2 * al(4 * n)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("nm,n", [((64, 64, 64), 5000), ((20, 30, 50), 1), ((100, 90, 80), (1 << 20) + 1)], ids=str)
def test_room_for_large_tiles_is_enough(nm, n, dtype):
    rng = np.random.default_rng(n)
    box = tuple(float(v) for v in nm)
    x = torch.tensor(rng.random((n, 3)) * nm, dtype=dtype, device="cuda")
    v = torch.tensor(rng.standard_normal((n, 3)), dtype=dtype, device="cuda")
    nb, flags = large_tile_bytes(nm, n), L.LDL_PAINT_FIXED
    assert nb < L.load().ldl_paint_workspace_bytes(L.i64x3(nm), 1, n, flags)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    one, three = torch.empty(nm, dtype=dtype, device="cuda"), torch.empty((3,) + nm, dtype=dtype, device="cuda")
    tail = (L.ptr(ws), nb, L.stream_ptr(x.device))
    L.call(f"ldl_ppaint_{L.sfx(dtype)}", L.ptr(x), L.pos_desc(box), n, None, 1.0, L.i64x3(nm), 1.0, flags, L.ptr(one), *tail)
    L.call(f"ldl_ppaint3D_{L.sfx(dtype)}", L.ptr(x), L.pos_desc(box), n, L.ptr(v), L.i64x3(nm), 1.0, flags, L.ptr(three), *tail)
    assert torch.equal(one, J.ppaint(x, 1.0, nm, box))
    assert torch.equal(three, J.ppaint3D(x, v, nm, box))
