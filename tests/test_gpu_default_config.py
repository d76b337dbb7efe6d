"""The default configuration (-1) over the sizes its rows-per-strip rule spans:
a strip of one row on the smallest domains, ragged last strips and rows, and
more strips than one round of resident waves.  Every configuration gives the
same bits, so the 2-D tile kernel is the reference."""

import ctypes

import numpy as np
import pytest

import helpers as H
from test_gpu_march_paths import _case

pytestmark = pytest.mark.gpu

TILE = 1


@pytest.mark.parametrize("nx,ny", [(2, 3), (61, 5), (96, 80), (503, 301), (1030, 517), (16, 8300), (5, 8193)])
@pytest.mark.parametrize("bc", [(1, 1, 1, 1), (2, 2, 2, 2), (1, 2, 1, 2)])
def test_default_equals_tile(nx, ny, bc):
    print("default config", nx, ny, bc, flush=True)
    inp, p, Hif, Hm = _case(nx, ny, bc, nx + ny, "land")
    D = H.DeviceDomain(inp)
    D.bathymetry_init()
    out = []
    for tile in (TILE, -1):
        h0, h1 = D.state(inp.eta, inp.hu, inp.hv), D.state(inp.eta, inp.hu, inp.hv)
        D.rk_steps(2, np.float32(0.3), h0, h1, tile=tile)
        out.append(D.host(h0))
    for a, b, name in zip(out[0], out[1], ("eta", "hu", "hv")):
        assert H.normal_equal(a, b), (name, H.diff_report(a, b))


def test_default_ensemble_equals_tile():
    print("default ensemble", flush=True)
    from SWESimulators import CDKLM16Ensemble, Common
    ctx = Common.HIPContext()
    members = []
    for k, (nx, ny, bc) in enumerate([(2, 2, (1, 1, 1, 1)), (64, 64, (1, 2, 1, 2)), (121, 33, (2, 2, 2, 2)), (59, 260, (2, 1, 2, 1))]):
        inp, _, _, _ = _case(nx, ny, bc, 40 + k, "deep")
        members.append(dict(nx=nx, ny=ny, dx=inp.dx, dy=inp.dy, f=inp.f, bc=bc, Hi=inp.Hi, eta=inp.eta, hu=inp.hu,
                            hv=inp.hv, wind_x=1e-4))
    states = []
    for cfg in (TILE, None):
        ens = CDKLM16Ensemble.CDKLM16Ensemble(ctx, members, dt=0.3, tile_config=cfg)
        ens.step_n(3)
        ens.gpu_stream.synchronize()
        states.append(ens.state[0].cpu().numpy())
        ens.cleanUp()
    assert H.normal_equal(*states)


@pytest.mark.parametrize("n,nx,ny,tile", [(1024, 16, 16, (16, 16)), (200, 16, 64, (16, 16)), (400, 32, 32, (32, 16)),
                                          (40, 16, 16, None), (300, 60, 16, None)])
def test_default_ensemble_of_small_members(n, nx, ny, tile):
    """Many small members take 2-D tiles by default, and give the bits of the
    marching kernel."""
    print("default small members", n, nx, ny, flush=True)
    from SWESimulators import CDKLM16Ensemble, Common, _gocean as G
    inp, _, _, _ = _case(nx, ny, (1, 2, 1, 2), n, "film")
    m = dict(nx=nx, ny=ny, dx=inp.dx, dy=inp.dy, f=inp.f, bc=inp.bc, Hi=inp.Hi, eta=inp.eta, hu=inp.hu, hv=inp.hv,
             wind_x=1e-4)
    states, tiles = [], []
    for cfg in (9, None):
        ens = CDKLM16Ensemble.CDKLM16Ensemble(Common.HIPContext(), [m] * n, dt=0.3, tile_config=cfg)
        ens.step_n(2)
        ens.gpu_stream.synchronize()
        count = ctypes.c_int()
        G.check(ens.lib.gocean_ensemble_info(ens.handle, None, ctypes.byref(count), None), "info")
        tiles.append(count.value)
        states.append(ens.state[0].cpu().numpy())
        ens.cleanUp()
    assert H.normal_equal(*states)
    assert tiles[1] == (tiles[0] if tile is None else n * -(-nx // tile[0]) * -(-ny // tile[1]))


@pytest.mark.parametrize("nx,ny", [(2, 2), (61, 5), (300, 1030)])
def test_max_dt_in_host_memory(nx, ny):
    """The minima the kernel writes to pinned host memory are the device's."""
    print("max dt host", nx, ny, flush=True)
    import torch
    inp, p, Hif, Hm = _case(nx, ny, (1, 2, 1, 2), nx, "film")
    D = H.DeviceDomain(inp)
    D.bathymetry_init()
    h = D.state(inp.eta, inp.hu, inp.hv)
    pinned = torch.zeros(2, pin_memory=True)
    D.G.check(D.lib.gocean_max_dt_host(D.dom, h[0].data_ptr(), h[1].data_ptr(), h[2].data_ptr(), D.Hm.data_ptr(), 0.7,
                                       D.scratch.data_ptr(), pinned.data_ptr(), None), "max_dt_host")
    torch.cuda.synchronize()
    got = pinned.numpy().copy()
    assert np.array_equal(got, D.scratch[:2].cpu().numpy())
    assert np.array_equal(got, D.max_dt(h, courant=0.7))
