"""Wave-uniform fast paths of the column-marching substep, bit for bit against
the CPU oracle.  A wavefront takes a fast path only when every used lane
qualifies, so the cases put the exceptions on single cells at the places where
a path can be chosen wrongly: the first and last columns of a strip (60 output
columns), the halo lanes, the first and last rows of a row strip, cells whose
depth straddles the desingularisation and the wet-face thresholds, single land
corners, and a land marker that lies among the depths."""

import numpy as np
import pytest

from oracle import cdklm16_np as O
import helpers as H

pytestmark = pytest.mark.gpu

MARCH8, MARCH_AUTO = 7, 9
BCS = [(1, 1, 1, 1), (2, 2, 2, 2), (1, 2, 1, 2)]
# depths around the switches: cutoff 1e-5, the wet-face limit
# (flux_eps / 2)^2 / g = 2.5e-4, desingularisation 0.1
FILMS = np.array([0.5e-5, 1.1e-5, 2.4e-4, 2.6e-4, 0.0999, 0.1001], np.float32)


class _Inp:
    pass


def _case(nx, ny, bc, seed, kind, dx=300.0, dy=250.0):
    rng = np.random.default_rng(seed)
    Hi = (20 + 5 * rng.random((ny + 5, nx + 5))).astype(np.float32)
    kw = {}
    spots = [(r, c) for r in (0, 1, ny // 2, ny - 1) for c in (0, 1, 57, 58, 59, 60, 61, 62, nx - 1) if c < nx]
    if kind == "land":
        for k, (r, c) in enumerate(spots):
            if k % 3 == 0:
                Hi[2 + r, 2 + c] = O.LAND_VALUE
    if kind == "marker":                      # a land value among the depths
        kw["land_value"] = 22.5
        Hi = np.where(np.abs(Hi - 22.5) < 0.01, np.float32(22.6), Hi)
        Hi[2 + ny // 2, 2:2 + nx:7] = 22.5
    p = O.Params(nx=nx, ny=ny, dx=dx, dy=dy, bc=bc, f=1.2e-4, **kw)
    Hif = O.bathymetry_halo(Hi, p)
    Hm = O.init_bm(Hif) if kind != "marker" else O.init_bm(Hif, land_value=22.5)
    eta = (0.3 * rng.standard_normal((ny + 4, nx + 4))).astype(np.float32)
    hu = (2 * rng.standard_normal(eta.shape)).astype(np.float32)
    hv = (2 * rng.standard_normal(eta.shape)).astype(np.float32)
    if kind == "film":
        for k, (r, c) in enumerate(spots):
            j, i = 2 + r, 2 + c
            eta[j, i] = -Hm[j, i] + FILMS[k % len(FILMS)]
            hu[j, i] *= 1e-4
            hv[j, i] *= 1e-4
    if kind != "marker":
        eta = np.maximum(eta, -Hm)
    O.periodic_bc(eta, hu, hv, p)
    inp = _Inp()
    inp.nx, inp.ny, inp.dx, inp.dy, inp.g, inp.r = nx, ny, dx, dy, 9.81, 0.0
    inp.bc, inp.f, inp.wind_x, inp.wind_y = bc, 1.2e-4, 1e-4, -2e-4
    p.wind_x, p.wind_y = (1e-4, 1e-4), (-2e-4, -2e-4)
    inp.Hi, inp.eta, inp.hu, inp.hv = Hi, eta, hu, hv
    return inp, p, Hif, Hm


@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 9), (57, 8), (60, 17), (61, 16), (64, 3), (121, 10)])
@pytest.mark.parametrize("bc", BCS)
@pytest.mark.parametrize("kind", ["deep", "film", "land"])
@pytest.mark.parametrize("rk", [0, 1])
def test_march_paths_bitexact(nx, ny, bc, kind, rk):
    print("march paths", nx, ny, bc, kind, rk, flush=True)
    inp, p, Hif, Hm = _case(nx, ny, bc, nx * 31 + ny, kind)
    D = H.DeviceDomain(inp)
    D.bathymetry_init()
    src = D.state(inp.eta, inp.hu, inp.hv)
    ref = O.cdklm_substep(0.4, rk, inp.eta, inp.hu, inp.hv, inp.eta, inp.hu, inp.hv, Hif, Hm, p)
    for tile in (MARCH8, MARCH_AUTO):
        dst = D.state(inp.eta, inp.hu, inp.hv)
        D.substep(0.4, rk, src, dst, tile=tile)
        for g, r_, name in zip(D.host(dst), ref, ("eta", "hu", "hv")):
            assert H.normal_equal(g[2:-2, 2:-2], r_[2:-2, 2:-2]), (tile, name, H.diff_report(g[2:-2, 2:-2], r_[2:-2, 2:-2]))


@pytest.mark.parametrize("dx,dy", [(1000.0 / 3.0, 77.7), (500.0, 123.456), (4.0, 2048.0), (1e-3, 1e5), (16777215.0, 3.0)])
def test_march_division_by_cell_size(dx, dy):
    """Cell sizes of many significands: whether or not the two-instruction
    division is exact for them, the result is the oracle's."""
    print("march division", dx, dy, flush=True)
    inp, p, Hif, Hm = _case(70, 23, (1, 2, 1, 2), 5, "deep", dx=dx, dy=dy)
    dt = np.float32(1e-3 * min(dx, dy))
    D = H.DeviceDomain(inp)
    D.bathymetry_init()
    src = D.state(inp.eta, inp.hu, inp.hv)
    dst = D.state(inp.eta, inp.hu, inp.hv)
    D.substep(dt, 0, src, dst, tile=MARCH8)
    ref = O.cdklm_substep(dt, 0, inp.eta, inp.hu, inp.hv, inp.eta, inp.hu, inp.hv, Hif, Hm, p)
    for g, r_, name in zip(D.host(dst), ref, ("eta", "hu", "hv")):
        assert H.normal_equal(g[2:-2, 2:-2], r_[2:-2, 2:-2]), (name, H.diff_report(g[2:-2, 2:-2], r_[2:-2, 2:-2]))


def test_march_land_marker_among_the_depths():
    """A land value inside the range of the depths: the fast path of the
    conversion is off, and the tile kernel agrees."""
    print("march land marker", flush=True)
    inp, p, Hif, Hm = _case(125, 21, (1, 1, 1, 1), 9, "marker")
    D = H.DeviceDomain(inp)
    D.dom.land_value = 22.5
    D.bathymetry_init()
    src = D.state(inp.eta, inp.hu, inp.hv)
    out = []
    for tile in (1, MARCH8, MARCH_AUTO):
        dst = D.state(inp.eta, inp.hu, inp.hv)
        D.substep(0.4, 0, src, dst, tile=tile)
        out.append(D.host(dst))
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)


SINGLE = [(4, 5), (10, 30), (15, 61), (12, 62), (17, 100), (8, 121)]
PAIRS = [(4, 5), (4, 6), (8, 20), (8, 22), (14, 40), (16, 40), (12, 60), (12, 62), (9, 100), (10, 100), (19, 121), (21, 121)]


MAX = float(np.finfo(np.float32).max)


@pytest.mark.parametrize("field,value", [(f, v) for f in ("eta", "hu", "hv", "Hi") for v in (np.nan, np.inf, -np.inf)]
                         + [("Hi", v) for v in (MAX, -MAX, 9.96921e36, -9.96921e36)])
@pytest.mark.parametrize("spots", [SINGLE, PAIRS], ids=["single", "pairs"])
def test_march_non_finite_cells(field, value, spots):
    """NaN and infinities, and the values files mark missing depths with, in
    single cells and in cells one or two apart in x or y, at a strip's inner
    columns and beside its edges: the marching kernel gives the 2-D tiles'
    result, NaN in the same cells and the same bits elsewhere, whatever the
    NaN's sign; cells whose stencil holds none of them are as if there were
    none, and momentum planted as NaN stays NaN."""
    print("march non-finite", field, value, flush=True)
    inp, p, Hif, Hm = _case(125, 21, (1, 1, 1, 1), 13, "deep", dx=100.0)
    runs = {}
    for sign in (1, -1):
        a = getattr(inp, field).copy()
        for r, c in spots:
            a[r, c] = np.copysign(np.float32(value), np.float32(sign)) if np.isnan(value) else value
        clean, at = getattr(inp, field), {field: a}
        for tile in (1, 5, MARCH8, MARCH_AUTO, -1):
            setattr(inp, field, at[field])
            D = H.DeviceDomain(inp)
            D.bathymetry_init()
            h0, h1 = D.state(inp.eta, inp.hu, inp.hv), D.state(inp.eta, inp.hu, inp.hv)
            D.substep(0.4, 0, h0, h1, tile=tile)
            runs[sign, tile] = np.stack(D.host(h1))[:, 2:-2, 2:-2]
            setattr(inp, field, clean)
    first = runs[1, 1]
    for key, got in runs.items():
        assert np.array_equal(first, got, equal_nan=True), key
    ref = np.stack(O.cdklm_substep(0.4, 0, inp.eta, inp.hu, inp.hv, inp.eta, inp.hu, inp.hv, Hif, Hm, p))[:, 2:-2, 2:-2]
    far = np.ones(ref.shape[1:], bool)
    for r, c in spots:
        far[max(0, r - 2 - 4):r - 2 + 5, max(0, c - 2 - 4):c - 2 + 5] = False
    assert far.any() and H.normal_equal(first[:, far], ref[:, far])
    if field in ("hu", "hv") and np.isnan(value):
        for r, c in spots:
            assert np.isnan(first[1:, r - 2, c - 2]).any(), (r, c)
