"""The 2-D tiles of the rotated and per-cell modes, bit for bit against the
oracle, where its shape and its second flux evaluation can go wrong: domains
smaller than a tile, one row or column past it, and north vectors that are the
same everywhere, differ in single cells, or differ everywhere."""

import ctypes

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


@pytest.mark.parametrize("nx,ny", [(505, 509), (9601, 8)])
def test_rotated_grid_of_many_tiles(nx, ny):
    """Sizes for which the 16x16 and the 32x8 tile are chosen."""
    print("rotated tiles", nx, ny, flush=True)
    test_rotated_grid_tile(nx, ny)


@pytest.mark.parametrize("mode", ["rotated", "field"])
@pytest.mark.parametrize("n,nx,ny,tile", [(300, 16, 16, (16, 16)), (300, 64, 8, (32, 8)), (600, 30, 13, (32, 14)),
                                          (300, 2, 5, (16, 16))])
def test_ensemble_general_tile(mode, n, nx, ny, tile):
    """An ensemble's tile follows its members' sizes, and each member's result
    is its own domain's."""
    print("ensemble general tile", mode, n, nx, ny, flush=True)
    import torch
    from SWESimulators import Common, _gocean as G
    lib = G.load()
    inp, p, _, _ = _case(nx, ny, (1, 2, 1, 2), 3, "film")
    north = (float(np.float32(np.sin(0.3))), float(np.float32(np.cos(0.3)))) if mode == "rotated" else (0.0, 1.0)
    rng = np.random.default_rng(5)
    ang = 0.4 * rng.random((ny + 4, nx + 4))
    fields = None if mode == "rotated" else ((1e-4 + 3e-5 * rng.random(ang.shape)).astype(np.float32),
                                             np.sin(ang).astype(np.float32), np.cos(ang).astype(np.float32))
    D = H.DeviceDomain(inp, north=north, fields=fields)
    D.bathymetry_init()
    plane = (ny + 4) * D.pitch
    members = (G.Member * n)()
    for k in range(n):
        members[k].domain = D.dom
        members[k].state_offset, members[k].hm_offset = 3 * k * plane, k * plane
        members[k].hi_offset = k * D.Hi.numel()
        members[k].field_offset = -1 if fields is None else 3 * k * plane
        members[k].wind.x0 = members[k].wind.x1 = inp.wind_x
        members[k].wind.y0 = members[k].wind.y1 = inp.wind_y
    handle = ctypes.c_void_p()
    G.check(lib.gocean_ensemble_create(members, n, -1, ctypes.byref(handle)), "ensemble_create")
    info = [ctypes.c_int() for _ in range(3)]
    G.check(lib.gocean_ensemble_info(handle, *[ctypes.byref(i) for i in info]), "info")
    state = [torch.stack(D.state(a, b, c)).repeat(n, 1, 1, 1).contiguous()
             for a, b, c in [(inp.eta, inp.hu, inp.hv)] * 2]
    Hi = D.Hi.repeat(n, 1, 1).contiguous()
    F = None if fields is None else torch.stack(D.field_t).repeat(n, 1, 1, 1).contiguous()
    dt = torch.full((n,), 0.4, device="cuda")
    G.check(lib.gocean_ensemble_substep(handle, 0, state[0].data_ptr(), None, state[1].data_ptr(), Hi.data_ptr(),
                                        None if F is None else F.data_ptr(), dt.data_ptr(), None), "ensemble_substep")
    dst = D.state(inp.eta, inp.hu, inp.hv)
    D.substep(0.4, 0, D.state(inp.eta, inp.hu, inp.hv), dst)
    torch.cuda.synchronize()
    want = torch.stack(dst).cpu().numpy()
    got = state[1].cpu().numpy()
    lib.gocean_ensemble_destroy(handle)
    for k in (0, 1, n // 2, n - 1):
        assert H.normal_equal(got[k][:, 2:-2, 2:nx + 2], want[:, 2:-2, 2:nx + 2]), k
    assert info[1].value == n * -(-nx // tile[0]) * -(-ny // tile[1])
