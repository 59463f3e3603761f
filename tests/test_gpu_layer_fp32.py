"""FP32 layers through the x passes of meshes with factors 3 and 5, forward and
backward, against the FP64 layer on the same positions (FP32 values, cells of
size one, so both see the same mesh coordinates): the fused pass at lengths on
both sides of its launch shapes with partial strips, and the separate passes
where the x axis is a power of two; and power-of-two meshes on every route of
the real-space stencils.  FP32 rounding is some 1e-6 of a norm here;
1e-4 is what a single wrong column of the largest mesh exceeds many times."""
import numpy as np
import pytest
import torch

from jerald_amd import _lib as L
from jerald_amd.model import JERALDModel
from jerald_amd.pmesh import PMesh

pytestmark = pytest.mark.gpu

MESHES = [(5, 8, 6), (45, 20, 30), (100, 12, 18), (360, 24, 20), (500, 16, 12), (972, 6, 10), (1000, 5, 6), (12, 96, 180), (64, 30, 20), (128, 16, 48)]
# columns enough for the shapes that fill the chip (more than 4096 in FP64, 8192 in FP32)
MANY = [(20, 96, 180), (240, 96, 180), (360, 64, 270), (640, 48, 180), (810, 60, 150), (960, 64, 144), (1000, 48, 180)]
# direct stencils up to 2^20 cells, marching ones 64, 256 and 128 (FP64 128) cells wide, partial tiles
POW2 = [(4, 8, 8), (64, 16, 1024), (32, 64, 1024), (1024, 8, 256), (64, 256, 1024), (1024, 128, 128)]
PRM = {"sm": [0.2, 0.7, 0.9, 4.0, 0.3], "dm": [0.2, 0.7, 0.9, 4.0, 0.3], "HI": [0.2, 0.7, 0.9, 4.0, 0.3, 0.1, 0.8, 1.1, 3.0, 0.2]}


def layer(nm, kind, dtype, X, star, v):
    m = JERALDModel(X.to(dtype), torch.zeros(nm), PMesh(nm, tuple(float(n) for n in nm), dtype=dtype), Nstep=1, kind=kind, starmap=star.to(dtype))
    out, rho, U, F, bins, S2 = m._layer_fwd(m.X, PRM[kind], 1.0, keep_bins=True)
    g, grad, ws = v.to(dtype).cuda(), torch.zeros(10, dtype=torch.float64, device="cuda"), m._ws()
    head = (L.ptr(m.X), m._pd(), X.shape[0], L.i64x3(nm), L.dvec(PRM[kind]), 1.0, 0, m.paint_flags)
    hi = (L.ptr(m.starmap), L.ptr(rho), L.ptr(U), L.ptr(S2)) if kind == "HI" else (L.ptr(rho), L.ptr(U))
    L.call(f"ldl_{kind.lower()}_layer_bwd_{L.sfx(dtype)}", *head, *hi, L.ptr(F), L.ptr(bins), L.ptr(g), L.ptr(g), L.ptr(grad), None, L.ptr(ws), ws.numel(),
           L.stream_ptr(g.device))
    return F.double(), g.double(), grad


@pytest.mark.parametrize("kind", ["sm", "dm", "HI"])
@pytest.mark.parametrize("nm", MESHES, ids=str)
def test_forces_and_adjoint_match_fp64(nm, kind):
    compare(nm, kind)


@pytest.mark.parametrize("kind", ["sm", "HI"])
@pytest.mark.parametrize("nm", MANY, ids=str)
def test_many_columns(nm, kind):
    compare(nm, kind)


@pytest.mark.parametrize("nm", POW2, ids=str)
def test_stencil_routes(nm):
    compare(nm, "sm")


def compare(nm, kind):
    rng = np.random.default_rng(21)
    q = np.stack(np.meshgrid(*[np.arange(n) for n in nm], indexing="ij"), -1).reshape(-1, 3)
    X = torch.tensor(np.mod(q + 0.4 * rng.standard_normal(q.shape), nm)).float()
    star, v = torch.tensor(rng.random(nm) + 0.1), torch.tensor(rng.standard_normal(q.shape)).float()
    for name, a, b in zip(("F", "g_in", "grad"), layer(nm, kind, torch.float32, X, star, v), layer(nm, kind, torch.float64, X, star, v)):
        assert torch.linalg.norm(a - b) <= 1e-4 * torch.linalg.norm(b), name
