"""The 2-D tile of the rotated and per-cell modes, bit for bit against the
oracle, where its shape and its second flux evaluation can go wrong: domains
smaller than a tile, one row or column past it, and north vectors that are the
same everywhere, differ in single cells, or differ everywhere."""

import numpy as np
import pytest

from oracle import cdklm16_np as O
import helpers as H
from test_gpu_march_paths import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2, 2), (31, 13), (32, 14), (33, 15), (70, 29)])
@pytest.mark.parametrize("bc", [(1, 1, 1, 1), (2, 2, 2, 2)])
@pytest.mark.parametrize("north", ["up", "rotated", "spots", "varying"])
def test_field_mode_tile(nx, ny, bc, north):
    print("field tile", nx, ny, bc, north, flush=True)
    inp, p, Hif, Hm = _case(nx, ny, bc, nx * 7 + ny, "land")
    rng = np.random.default_rng(nx)
    shape = (ny + 4, nx + 4)
    ang = {"up": np.zeros(shape), "rotated": np.full(shape, 0.4), "spots": np.zeros(shape),
           "varying": 0.4 * rng.random(shape)}[north]
    if north == "spots":
        ang[::5, ::6] = 0.7
    f = (1e-4 + 3e-5 * rng.random(shape)).astype(np.float32)
    fields = (f, np.sin(ang).astype(np.float32), np.cos(ang).astype(np.float32))
    p.f, p.north_x, p.north_y = fields
    D = H.DeviceDomain(inp, fields=fields)
    D.bathymetry_init()
    src = D.state(inp.eta, inp.hu, inp.hv)
    for rk in (0, 1):
        dst = D.state(inp.eta, inp.hu, inp.hv)
        D.substep(0.4, rk, src, dst)
        ref = O.cdklm_substep(0.4, rk, inp.eta, inp.hu, inp.hv, inp.eta, inp.hu, inp.hv, Hif, Hm, p)
        for g, r_, name in zip(D.host(dst), ref, ("eta", "hu", "hv")):
            assert H.normal_equal(g[2:-2, 2:-2], r_[2:-2, 2:-2]), (name, H.diff_report(g[2:-2, 2:-2], r_[2:-2, 2:-2]))


@pytest.mark.parametrize("nx,ny", [(31, 13), (33, 29)])
def test_rotated_grid_tile(nx, ny):
    print("rotated tile", nx, ny, flush=True)
    inp, p, Hif, Hm = _case(nx, ny, (1, 2, 1, 2), nx + ny, "film")
    north = (float(np.float32(np.sin(0.3))), float(np.float32(np.cos(0.3))))
    p.north_x, p.north_y = north
    D = H.DeviceDomain(inp, north=north)
    D.bathymetry_init()
    src = D.state(inp.eta, inp.hu, inp.hv)
    dst = D.state(inp.eta, inp.hu, inp.hv)
    D.substep(0.4, 0, src, dst)
    ref = O.cdklm_substep(0.4, 0, inp.eta, inp.hu, inp.hv, inp.eta, inp.hu, inp.hv, Hif, Hm, p)
    for g, r_, name in zip(D.host(dst), ref, ("eta", "hu", "hv")):
        assert H.normal_equal(g[2:-2, 2:-2], r_[2:-2, 2:-2]), (name, H.diff_report(g[2:-2, 2:-2], r_[2:-2, 2:-2]))
