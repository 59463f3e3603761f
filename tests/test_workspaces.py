"""Workspace sizes by position form (CPU): lattice positions pay for the sort's
keys and indices alone, absolute ones for its lists too, which in a layer lie
in the spectra's room."""
import pytest

from jerald_amd import _lib as L


def sort_bytes(nm, n):
    tiles = -(-nm[0] // 8) * -(-nm[1] // 16) * -(-nm[2] // 16)  # three components may take flat tiles
    return 8 * n + 64 * tiles + (1 << 16)


@pytest.mark.parametrize("side", [512, 1024])
@pytest.mark.parametrize("nc", [1, 3])
def test_paint_of_lattice_positions_has_no_lists(side, nc):
    nm, n = (side,) * 3, side**3
    q = L.load().ldl_paint_workspace_bytes
    lists = q(L.i64x3(nm), nc, n, 0) - q(L.i64x3(nm), nc, n, L.LDL_PAINT_LATTICE)
    assert q(L.i64x3(nm), nc, n, L.LDL_PAINT_LATTICE) <= sort_bytes(nm, n)
    assert 12 * n <= lists <= 12 * n + (10 << 20)
    direct = L.LDL_PAINT_DIRECT  # does not sort
    assert q(L.i64x3(nm), nc, n, direct) == q(L.i64x3(nm), nc, n, direct | L.LDL_PAINT_LATTICE) <= sort_bytes(nm, n) + 8 * nc * n + (1 << 16)


@pytest.mark.parametrize("side", [256, 512, 1024])
@pytest.mark.parametrize("f64", [0, 1])
def test_layer_holds_the_lists_in_its_spectra(side, f64):
    nm, n, b = (side,) * 3, side**3, 4 << f64
    q = L.load().ldl_sm_workspace_bytes
    pitch = L.load().ldl_sm_spectrum_pitch(L.i64x3(nm), f64)
    rest = sort_bytes(nm, n) + 3 * side**2 * pitch * 2 * b + 3 * n * b + 12 * 8 * (2 * side**2 + side * (side // 2 + 2) + 4096) + (1 << 16)
    assert q(L.i64x3(nm), f64, n, 0) <= rest
    # eight particles a cell: the spectra hold no more, absolute positions add the rest
    assert q(L.i64x3(nm), f64, 8 * n, L.LDL_PAINT_LATTICE) <= rest + 8 * 7 * n
    assert q(L.i64x3(nm), f64, 8 * n, 0) > rest + 8 * 7 * n
