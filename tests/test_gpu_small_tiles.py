"""The paint's tile sizes and the sort's chunk size at the lines where they
change, on meshes with partial and short tiles.  The fixed-point paint gives
the same bits for every split, so each case is compared with the CPU
emulation of it."""
import numpy as np
import pytest
import torch

from jerald_amd import _lib as L
from jerald_amd import jaxpops as J
from oracle import native as NV

pytestmark = pytest.mark.gpu

# 64-bit three-component sums and FP64 take flat tiles (8 x 16 x 16) from 256
# large tiles on.  255 and 256 large tiles (8 x 16 x 32 cells), one cell, sides below and just
# above a small tile's (4 x 8 x 16); particle numbers around 512, 2048 and the
# two lines
CASES = [((40, 272, 96), 513), ((32, 256, 128), 512), ((64, 64, 256), 2049), ((1, 1, 1), 3), ((3, 7, 15), 511), ((5, 9, 17), 2047),
         ((2, 8, 64), 1), ((33, 257, 113), 40000), ((64, 144, 240), 4097), ((37, 53, 70), (1 << 20) - 1), ((64, 32, 48), 1 << 20), ((20, 20, 20), (1 << 22) - 1), ((20, 20, 20), 1 << 22)]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("nm,n", CASES, ids=lambda v: str(v))
def test_paint_bits_for_any_split(nm, n, dtype):
    rng = np.random.default_rng(n)
    box = tuple(float(v) for v in nm)
    x = np.mod(rng.random((n, 3)) * nm, nm).astype(dtype)
    got = J.ppaint(torch.tensor(x, device="cuda"), 1.0, nm, box).cpu().numpy()
    acc, s = NV.paint_fixed(x, 1.0, nm, box=box, dtype=dtype)
    assert np.array_equal(got, NV.fixed_to_float(acc, s, np.dtype(dtype).type))
    m = rng.standard_normal((n, 3)).astype(dtype)
    got = J.ppaint3D(torch.tensor(x, device="cuda"), torch.tensor(m, device="cuda"), nm, box).cpu().numpy()
    for c in range(3):
        acc, s = NV.paint_fixed(x, np.ascontiguousarray(m[:, c]), nm, box=box, dtype=dtype)
        assert np.array_equal(got[c], NV.fixed_to_float(acc, s, np.dtype(dtype).type)), c


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_three_components_without_room_for_flat_tiles(dtype):
    # the query's bytes less the keys that the flat tiles have beyond the large ones
    n, nm = 5000, (64, 256, 128)
    box = tuple(float(v) for v in nm)
    rng = np.random.default_rng(3)
    x = torch.tensor(rng.random((n, 3)) * nm, dtype=dtype, device="cuda")
    v = torch.tensor(rng.standard_normal((n, 3)), dtype=dtype, device="cuda")
    nb = L.load().ldl_paint_workspace_bytes(L.i64x3(nm), 3, n, L.LDL_PAINT_FIXED) - 8 * 512 * 8
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    out = torch.empty((3,) + nm, dtype=dtype, device="cuda")
    L.call(f"ldl_ppaint3D_{L.sfx(dtype)}", L.ptr(x), L.pos_desc(box), n, L.ptr(v), L.i64x3(nm), 1.0, L.LDL_PAINT_FIXED, L.ptr(out), L.ptr(ws), nb,
           L.stream_ptr(x.device))
    assert torch.equal(out, J.ppaint3D(x, v, nm, box))
