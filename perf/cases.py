"""Timed cases of the CDKLM16 framework: single-domain steps, batched
ensembles (plain and with model error and drifters), reverse mode and the
localised analysis, through the public Python classes.

A case is a dict of plain values; ``kind`` says which entry point it takes:

  step   CDKLM16.step_n / CDKLM16.step on one domain
  ens    CDKLM16Ensemble.step_n on many domains
  adj    adjoint.CDKLM16RK2.apply and its backward on one domain
  ensadj EnsembleAdjoint.forward / backward on domains of several sizes
  letkf  ETKFOcean.LETKF on an ensemble

``exact`` evaluates the same scheme in float64 with plain torch operations.
"""

import math
import os
import sys

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "gpu-ocean_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "gpu-ocean_amd"))

GRAV, F0, BETA, THETA = 9.81, 1.2e-4, 2.0e-11, 1.3
LAND = float(np.float32(1.0e20))
DESING, FLUX_EPS, CUTOFF, DRY = 1.0e-1, 1.0e-1, 1.0e-5, 1.0e-30
Q0 = 2.0e-5                     # amplitude of the model error, metres
F64 = torch.float64
WALL, PERIODIC = 1, 2


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a regional pilot run or one particle of a small filter: a few
        # thousand cells, one model step a call, so launches are what counts
        dict(name="step-96x80", kind="step", nx=96, ny=80, steps=1, ns=False, ew=False),
        # a coastal domain of odd sides with a masked coast, shoals and a
        # gridded wind field
        dict(name="step-coast-503x301", kind="step", nx=503, ny=301, steps=10, ns=False, ew=False,
             coast=True, wind="grid"),
        # the step loop as an application drives it: simulated seconds, dt
        # from the CFL condition before every step, doubly periodic
        dict(name="step-cfl-500x300", kind="step", nx=500, ny=300, steps=6, ns=True, ew=True, cfl=True),
        # beta plane: the Coriolis parameter is a field
        dict(name="step-beta-640x417", kind="step", nx=640, ny=417, steps=10, ns=False, ew=True, beta=True),
        # the headline domain of bench.py
        dict(name="step-2048x2048", kind="step", nx=2048, ny=2048, steps=10, ns=False, ew=True,
             wind="uniform"),
        # many small members
        dict(name="ens-1024x64x64", kind="ens", members=1024, nx=64, ny=64, steps=5, ns=False, ew=False),
        # the ensemble of bench.py
        dict(name="ens-100x512x512", kind="ens", members=100, nx=512, ny=512, steps=2, ns=False, ew=False),
        # a forecast of the data-assimilation cycle on the double-jet domain:
        # every step with model error and drifters, then the observations
        dict(name="ens-forecast-100x500x300", kind="ens", members=100, nx=500, ny=300, steps=3, ns=False,
             ew=True, noise=1, drifters=64),
        # gradient of a point misfit with respect to the initial state
        dict(name="adj-512x512", kind="adj", nx=512, ny=512, steps=25, ns=False, ew=False),
        # the same for the domains of a multi-domain problem at once
        dict(name="ensadj-16", kind="ensadj", domains=16, steps=6),
        # localised analysis of the double-jet ensemble, a buoy every 25 cells
        dict(name="letkf-100x500x300", kind="letkf", members=100, nx=500, ny=300, every=25),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "ens", "ens", "adj", "ensadj", "letkf"])
    ns, ew = rng.random() < 0.4, rng.random() < 0.5
    if kind == "step":
        c = dict(kind=kind, nx=_side(rng, 24, 2048), ny=_side(rng, 24, 2048), steps=rng.randint(1, 10), ns=ns, ew=ew,
                 wind=rng.choice(["none", "uniform", "grid"]))
        extra = rng.choice(["", "", "coast", "cfl", "beta"])
        if extra:
            c[extra] = True
        return c
    if kind == "ens":
        nx, ny = _side(rng, 40, 512), _side(rng, 40, 512)
        most = max(2, min(1024, 26_000_000 // (nx * ny)))
        c = dict(kind=kind, members=_side(rng, 2, most), nx=nx, ny=ny, steps=rng.randint(1, 3), ns=ns, ew=ew)
        if rng.random() < 0.5:
            c["noise"] = rng.choice([1, 1, 3, 5])
            c["drifters"] = rng.choice([0, 16, 64])
            c["nx"], c["ny"] = (max(c["noise"] * 9, n - n % c["noise"]) for n in (nx, ny))
        return c
    if kind == "adj":
        return dict(kind=kind, nx=_side(rng, 48, 900), ny=_side(rng, 48, 900), steps=rng.randint(3, 15), ns=ns, ew=ew)
    if kind == "ensadj":
        return dict(kind=kind, domains=rng.randint(2, 16), steps=rng.randint(2, 6))
    nx, ny = rng.randint(80, 500), rng.randint(80, 300)
    return dict(kind=kind, members=rng.randint(10, 100), nx=nx, ny=ny, every=rng.choice([25, 25, 40, 50]))


def _cells(c):
    if c["kind"] == "ensadj":
        return sum(nx * ny for nx, ny in _sides(c))
    return c.get("members", 1) * c["nx"] * c["ny"]


def work(case):
    """A step reads the state and the corner depths and writes the state once
    (28 B a cell) and takes about 330 operations a cell and stage.  Reverse
    mode takes the step and about three times its operations again, and reads
    and writes the adjoint.  The analysis reads and writes the cells under a
    weight."""
    n = _cells(case)
    if case["kind"] == "letkf":
        r = _letkf_r(case)
        buoys = -(-case["nx"] // case["every"]) * -(-case["ny"] // case["every"])
        cells = buoys * math.pi * (1.5 * r) ** 2
        return {"bytes": 24.0 * case["members"] * min(cells, 8 * case["nx"] * case["ny"]),
                "flops": 2.0 * 3 * cells * case["members"] ** 2}
    steps = case["steps"]
    if case["kind"] in ("adj", "ensadj"):
        return {"bytes": 28.0 * n + 28.0 * n + 56.0 * n * (steps - 1), "flops": 660.0 * 4 * n * steps}
    more = 28.0 * n * steps if case.get("noise") else 0.0
    return {"bytes": 28.0 * n * steps + more, "flops": 660.0 * n * steps}


def tolerance(case):
    """About four times what the path is off from ``exact``: float32 rounding
    acts on the water depth, so the transports of a deep, slow ocean are off
    by more than their own last bits; the reverse mode takes the branches of
    its own forward, and some differ in 64 bits."""
    if case["kind"] in ("adj", "ensadj"):
        return {"rel": 2e-2, "max": 0.9}
    if case["kind"] == "letkf":
        return {"rel": 1e-6, "max": 1e-4}
    if case["kind"] == "ens":
        return {"rel": 2e-5, "max": 5e-3}
    return {"rel": 2e-4, "max": 5e-2}


# ---------------------------------------------------------------------------
# inputs, made from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _smooth(g, n, ny, nx, corr):
    """n periodic random fields of unit variance with Gaussian correlation of
    ``corr`` cells."""
    noise = torch.randn((n, ny, nx), generator=g, device="cuda")
    ky = torch.fft.fftfreq(ny, device="cuda")[:, None]
    kx = torch.fft.rfftfreq(nx, device="cuda")[None, :]
    filt = torch.exp(-0.25 * (2 * math.pi) ** 2 * (kx ** 2 + ky ** 2) * corr ** 2)
    a = torch.fft.irfft2(torch.fft.rfft2(noise) * filt, s=(ny, nx))
    a = a - a.mean(dim=(1, 2), keepdim=True)
    return a / a.std(dim=(1, 2), keepdim=True).clamp_min(1e-12)


def _balanced(eta, Hi, dx):
    """Transports in geostrophic balance with eta."""
    Hm = 0.25 * (Hi[..., :-1, :-1] + Hi[..., 1:, :-1] + Hi[..., :-1, 1:] + Hi[..., 1:, 1:])
    h = eta + Hm
    hu, hv = torch.zeros_like(eta), torch.zeros_like(eta)
    k = GRAV / F0 / (2 * dx)
    hu[..., 1:-1, :] = -k * h[..., 1:-1, :] * (eta[..., 2:, :] - eta[..., :-2, :])
    hv[..., :, 1:-1] = k * h[..., :, 1:-1] * (eta[..., :, 2:] - eta[..., :, :-2])
    return hu, hv


def _chart(Hi):
    """Depths in steps of 1/64 m, as charts give them: a cell and its mirror
    image behind a wall then have the same depth in any precision, and the
    upwind choice at the wall, where the normal velocities cancel, is no
    matter of rounding."""
    return torch.where(Hi > LAND / 2, Hi, torch.round(Hi * 64) / 64).float()


def _domain(case, seed, members, nx, ny, dx):
    """(eta, hu, hv, Hi) of ``members`` domains as float32 device tensors."""
    g = _gen(seed)
    if case.get("coast"):
        # shoals off a straight masked coast
        Hi = 12.0 + 14.0 * _smooth(g, 1, ny + 5, nx + 5, 20.0)[0]
        Hi = Hi.clamp_min(1.0)
        Hi[:2 + max(2, ny // 8)] = LAND
        eta = 0.08 * _smooth(g, members, ny + 4, nx + 4, 12.0)
        z = torch.zeros_like(eta)
        return eta.float(), z, z.clone(), _chart(Hi)
    if case["kind"] == "letkf" or case.get("drifters") is not None:
        Hi = torch.full((ny + 5, nx + 5), 1000.0, device="cuda")          # double jet
        row = torch.arange(ny + 4, device="cuda", dtype=torch.float32)[:, None]
        w = 0.04 * ny
        jet = torch.exp(-((row - ny / 4) / w) ** 2) - torch.exp(-((row - 3 * ny / 4) / w) ** 2)
        eta = 0.3 * jet + 0.02 * _smooth(g, members, ny + 4, nx + 4, 8.0)
    else:
        Hi = (100.0 + 30.0 * _smooth(g, 1, ny + 5, nx + 5, 32.0)[0]).clamp_min(10.0)
        eta = 0.15 * _smooth(g, 1, ny + 4, nx + 4, 24.0) + 0.05 * _smooth(g, members, ny + 4, nx + 4, 16.0)
    Hi = _chart(Hi)
    hu, hv = _balanced(eta, Hi, dx)
    return eta.float(), hu.float(), hv.float(), Hi


def _dx(case):
    return 2000.0 if case["kind"] == "letkf" or case.get("drifters") is not None else 500.0


def _dt(Hi, dx):
    """A step of CFL number 0.6 for water of this depth, as a float32."""
    deep = float(Hi[Hi < LAND / 2].max())
    return float(np.float32(0.6 * 0.25 * dx / (math.sqrt(GRAV * (deep + 1.0)) + 2.0)))


def _bc(case):
    ns, ew = (PERIODIC if case.get(k) else WALL for k in ("ns", "ew"))
    return ns, ew, ns, ew


def _wind(case, seed):
    """(X, Y) fields of the wind stress, float32 host arrays."""
    kind = case.get("wind", "none")
    if kind == "grid":
        rs = np.random.RandomState(seed & 0xFFFF)
        return tuple((1e-4 * rs.standard_normal((7, 11))).astype(np.float32) for _ in range(2))
    a = 0.1 / 1025.0 if kind == "uniform" else 0.0
    return tuple(np.array([[a * b]], np.float32) for b in (math.cos(math.pi / 6), math.sin(math.pi / 6)))


def _sides(case):
    """Sides of a multi-domain problem."""
    return [(256 + 128 * ((5 * k) % 5 + k % 3) - 3 * (k % 2), 256 + 64 * ((3 * k) % 7)) for k in range(case["domains"])]


def _letkf_r(case):
    """Localisation scale in cells, as large as the buoys' spacing allows."""
    return min(15.0, math.floor(min(case["nx"], case["ny"]) / 5.0))


def _buoys(case, seed):
    ys, xs = np.mgrid[0:case["ny"]:case["every"], 0:case["nx"]:case["every"]]
    dx = _dx(case)
    rs = np.random.RandomState(seed & 0xFFFFFF)
    n = xs.size
    return np.column_stack([(xs.ravel() + 0.5) * dx, (ys.ravel() + 0.5) * dx, 5.0 * rs.standard_normal((n, 2))])


def _points(nx, ny, dx, seed, n):
    rs = np.random.RandomState((seed * 7 + nx) & 0xFFFFFF)
    return rs.uniform(3.0, nx - 3.0, n) * dx, rs.uniform(3.0, ny - 3.0, n) * dx, (0.1 * rs.standard_normal(n)).astype(np.float32)


# ---------------------------------------------------------------------------
# the framework
# ---------------------------------------------------------------------------
_CTX = []


def _ctx():
    from SWESimulators import Common
    if not _CTX:
        _CTX.append(Common.HIPContext())
    return _CTX[0]


def _simulator(case, seed):
    from SWESimulators import CDKLM16, Common, WindStress
    nx, ny, dx = case["nx"], case["ny"], _dx(case)
    eta, hu, hv, Hi = _domain(case, seed, 1, nx, ny, dx)
    X, Y = _wind(case, seed)
    return CDKLM16.CDKLM16(_ctx(), eta[0].cpu().numpy(), hu[0].cpu().numpy(), hv[0].cpu().numpy(), Hi.cpu().numpy(),
                           nx, ny, dx, dx, _dt(Hi, dx), GRAV, F0, 0.0,
                           coriolis_beta=BETA if case.get("beta") else 0.0, courant_number=0.6,
                           boundary_conditions=Common.BoundaryConditions(*_bc(case)),
                           wind_stress=WindStress.WindStress(t=[0.0], X=[X], Y=[Y]))


def _ensemble(case, seed):
    from SWESimulators import CDKLM16Ensemble
    dx = _dx(case)
    if case["kind"] == "ensadj":
        parts = [(nx, ny, _domain(case, seed * 31 + k, 1, nx, ny, dx)) for k, (nx, ny) in enumerate(_sides(case))]
        doms = [(nx, ny, [a[0].cpu().numpy() for a in p[:3]], p[3].cpu().numpy(), _dt(p[3], dx)) for nx, ny, p in parts]
    else:
        nx, ny = case["nx"], case["ny"]
        eta, hu, hv, Hi = _domain(case, seed, case["members"], nx, ny, dx)
        state, hi, dt = [a.cpu().numpy() for a in (eta, hu, hv)], Hi.cpu().numpy(), _dt(Hi, dx)
        doms = [(nx, ny, [a[k] for a in state], hi, dt) for k in range(case["members"])]
    members = [dict(nx=nx, ny=ny, dx=dx, dy=dx, g=GRAV, f=F0, bc=_bc(case), Hi=hi, eta=q[0], hu=q[1], hv=q[2])
               for nx, ny, q, hi, _ in doms]
    ens = CDKLM16Ensemble.CDKLM16Ensemble(_ctx(), members, dt=[d[4] for d in doms])
    if case.get("noise"):
        ens.enable_model_error(soar_q0=Q0, interpolation_factor=case["noise"], seed=seed & 0xFFFFFF)
    if case.get("drifters"):
        ens.enable_drifters(case["drifters"])
    return ens


def _misfit_setup(shapes, offsets, dx, seed):
    """Stencils and data of 64 points a domain in one flat state."""
    from SWESimulators import adjoint
    idx, wt, ys = [], [], []
    for k, ((nx, ny), off) in enumerate(zip(shapes, offsets)):
        ox, oy, y = _points(nx, ny, dx, seed + k, 64)
        i, w = adjoint.bilinear_stencil(int(off), nx + 4, ox, oy, dx, dx)
        idx.append(i), wt.append(w), ys.append(y)
    return tuple(torch.from_numpy(np.concatenate(a)).cuda() for a in (idx, wt, ys))


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("step", "adj"):
        sim = s["sim"] = _simulator(case, seed)
        s["t_end"] = case["steps"] * sim.dt * 0.97
    else:
        ens = s["ens"] = _ensemble(case, seed)
    if kind == "adj":
        from SWESimulators import adjoint
        s["adj"] = adjoint.simulator_adjoint(sim)
        s["q0"] = [a.tensor.clone() for a in (sim.gpu_data.h0, sim.gpu_data.hu0, sim.gpu_data.hv0)]
        s["misfit"] = _misfit_setup([(case["nx"], case["ny"])], [0], _dx(case), seed)
    elif kind == "ensadj":
        from SWESimulators import adjoint
        s["adj"] = adjoint.EnsembleAdjoint(ens)
        s["q0"] = ens.state[0].clone()
        s["misfit"] = _misfit_setup(_sides(case), ens.state_off[:-1], _dx(case), seed)
    elif kind == "letkf":
        from SWESimulators import ETKFOcean
        s["filter"] = ETKFOcean.ETKFOcean(ens, np.diag([1.0, 1.0]))
        s["obs"] = _buoys(case, seed)
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "step":
        sim = s["sim"]
        if case.get("cfl"):
            sim.step(s["t_end"], update_dt=True)
        else:
            sim.step_n(case["steps"])
        return {"eta": sim.gpu_data.h0.tensor, "hu": sim.gpu_data.hu0.tensor, "hv": sim.gpu_data.hv0.tensor}
    if kind == "ens":
        ens = s["ens"]
        ens.step_n(case["steps"], model_error=bool(case.get("noise")))
        out = {"state": ens.state[0]}
        if case.get("drifters"):
            out["observed"] = ens.observe()
            out["drifters"] = ens.drifter_positions[:, :case["drifters"]]
        return out
    if kind == "adj":
        from SWESimulators import adjoint
        idx, wt, y = s["misfit"]
        q = [a.detach().requires_grad_(True) for a in s["q0"]]
        out = adjoint.CDKLM16RK2.apply(*q, s["adj"], case["steps"], s["sim"].dt)
        J = adjoint.stencil_misfit(out[0].reshape(-1), idx, wt, y)
        J.backward()
        return {"J": J.detach(), "state": [a.detach() for a in out], "grad": [a.grad for a in q]}
    if kind == "ensadj":
        from SWESimulators import adjoint
        idx, wt, y = s["misfit"]
        out = s["adj"].forward(s["q0"], case["steps"]).requires_grad_(True)
        J = adjoint.stencil_misfit(out, idx, wt, y)
        lam = torch.autograd.grad(J, out)[0]
        return {"J": J.detach(), "state": out.detach(), "grad": s["adj"].backward(lam)}
    s["filter"].LETKF(s["obs"], r_factor=_letkf_r(case))
    return {"state": s["ens"].state[0]}


# ---------------------------------------------------------------------------
# the same in float64, with plain torch operations
# ---------------------------------------------------------------------------
def _ghosts(n, periodic):
    """Source index and sign of the normal transport of each padded index."""
    i = torch.arange(n + 4, device="cuda")
    sg = torch.ones(n + 4, dtype=F64, device="cuda")
    if periodic:
        return (i - 2) % n + 2, sg
    src = torch.where(i < 2, 3 - i, torch.where(i > n + 1, 2 * n + 3 - i, i))
    sg[:2] = -1.0
    sg[-2:] = -1.0
    return src, sg


def _halo(Hi, nx, ny, ns, ew):
    """Corner depths with their halo completed, north-south first."""
    def fill(n, periodic):
        i = torch.arange(n + 5, device="cuda")
        if periodic:
            return torch.where(i < 2, i + n, torch.where(i > n + 1, i - n, i))
        return torch.where(i < 2, 4 - i, torch.where(i > n + 2, 2 * n + 4 - i, i))
    return Hi.double()[..., fill(ny, ns), :][..., :, fill(nx, ew)]


def _minmod(a, b, c):
    pos = torch.minimum(torch.minimum(a, b), c).clamp_min(0.0)
    return pos + torch.maximum(torch.maximum(a, b), c).clamp_max(0.0)


def _upwind(hm, um, vm, hp, up, vp):
    """Central-upwind flux between the states m and p; u is along the face's
    normal."""
    wm, wp = hm > CUTOFF, hp > CUTOFF
    z = torch.zeros_like(hm)
    one = torch.ones_like(hm)

    def side(w, h, u, v):
        q = h * u
        c = torch.sqrt(GRAV * torch.where(w, h, one))
        return [torch.where(w, a, z) for a in (q, q * u + 0.5 * GRAV * h * h, q * v, u, c)]

    m0, m1, m2, su, sc = side(wm, hm, um, vm)
    p0, p1, p2, tu, tc = side(wp, hp, up, vp)
    lo = torch.minimum(torch.minimum(su - sc, tu - tc), z)
    hi = torch.maximum(torch.maximum(su + sc, tu + tc), z)
    still = (hi - lo).abs() < FLUX_EPS
    den = torch.where(still, one, hi - lo)
    f0 = (hi * m0 - lo * p0 + hi * lo * (hp - hm)) / den
    f1 = (hi * m1 - lo * p1 + hi * lo * (p0 - m0)) / den
    f2 = torch.where(um + up > 0, m2, p2)
    return [torch.where(still, z, f) for f in (f0, f1, f2)]


def _axis_fluxes(E, a, b, Hlo, Hhi, dry, flip, flip_adj, sg, f, d):
    """Along the last axis, for cells 1 .. n+2 of n+4: the geostrophic slope
    term T of every interior cell and the fluxes of the n+1 faces between
    cells 1 .. n+2.  a is the velocity along the axis, b the one across it;
    sg is -1 on the x axis (K = g eta_x - f v) and +1 on the y axis."""
    def at(x, k):
        n = x.shape[-1]
        return x[..., k:n - 2 + k]

    def slope(x):
        return _minmod((at(x, 1) - at(x, 0)) * THETA, (at(x, 2) - at(x, 0)) * 0.5, (at(x, 2) - at(x, 1)) * THETA)

    fb = f * b * flip
    k = d / (2 * GRAV) * sg
    l, c, r = at(fb, 0), at(fb, 1), at(fb, 2)
    e = at(E, 1)
    K = _minmod(THETA * GRAV * (e - at(E, 0) + k * (c + l)), 0.5 * GRAV * (at(E, 2) - at(E, 0) + k * (r + 2 * c + l)),
                THETA * GRAV * (at(E, 2) - e + k * (c + r)))
    lo, hi = at(Hlo, 1), at(Hhi, 1)
    adj = -sg * d * at(f * b * flip_adj, 1)
    t = (K + adj) / (2 * GRAV)
    low, high = e + lo - t <= 0, e + hi + t <= 0
    K = torch.where(low, -adj + 2 * GRAV * (e + lo), K)
    K = torch.where(high, -adj - 2 * GRAV * (e + hi), K)
    T = (K - sg * d * at(fb, 1)) / (2 * GRAV)
    sa, sb = slope(a), slope(b)
    ac, bc, w = at(a, 1), at(b, 1), at(dry, 1)
    m, p = (slice(None, -1), slice(1, None))
    hm = (e + hi + T)[..., m].clamp_min(0.0)
    hp = (e + lo - T)[..., p].clamp_min(0.0)
    F = _upwind(hm, (ac + 0.5 * sa)[..., m], (bc + 0.5 * sb)[..., m], hp, (ac - 0.5 * sa)[..., p], (bc - 0.5 * sb)[..., p])
    closed = w[..., m] | w[..., p]
    return T[..., 1:-1], [torch.where(closed, torch.zeros_like(x), x) for x in F]


class _Scheme:
    """One domain (or members that share one) of the scheme in float64."""

    def __init__(self, case, nx, ny, dx, Hi, X=0.0, Y=0.0):
        ns, ew = bool(case.get("ns")), bool(case.get("ew"))
        self.nx, self.ny, self.dx, self.X, self.Y, self.ns, self.ew = nx, ny, dx, X, Y, ns, ew
        self.rows, self.sv = _ghosts(ny, ns)
        self.cols, self.su = _ghosts(nx, ew)
        # the sign of the tangential velocity in the geostrophic terms, and
        # the one the positivity adjustment takes (low walls only)
        self.fx, self.fy = self.su, self.sv
        self.ax, self.ay = self.su.clone(), self.sv.clone()
        self.ax[-2:] = 1.0
        self.ay[-2:] = 1.0
        H = _halo(Hi, nx, ny, ns, ew)
        H = torch.where((H - LAND).abs() < 1e-3, torch.full_like(H, DRY), H)
        a, b, c, d = H[:-1, :-1], H[1:, :-1], H[:-1, 1:], H[1:, 1:]
        wet = sum((x != DRY).double() for x in (a, b, c, d))
        self.land = wet == 0
        self.Hm = torch.where(self.land, torch.zeros_like(a), (a + b + c + d) / wet.clamp_min(1.0))
        self.Hc = 0.25 * (a + b + c + d)
        self.W, self.Ea, self.S, self.N = (0.5 * x for x in (a + b, c + d, a + c, b + d))
        f = torch.full((ny + 4,), float(np.float32(F0)), dtype=F64, device="cuda")
        if case.get("beta"):
            f = F0 - 2 * BETA * dx + BETA * (torch.arange(ny + 4, device="cuda", dtype=F64) - 1.5) * dx
        self.f = f[:, None]

    def stage(self, e, hu, hv, dt, qn=None):
        e = e[..., self.rows, :][..., :, self.cols]
        hu = hu[..., self.rows, :][..., :, self.cols] * self.su
        hv = hv[..., self.rows, :][..., :, self.cols] * self.sv[:, None]
        h = e + self.Hm
        z = torch.zeros_like(h)
        dry = (~self.land) & (h <= CUTOFF)
        thin = (~self.land) & (h < DESING) & ~dry
        closed = self.land | dry
        hd = torch.where(closed, torch.ones_like(h), h)
        den = torch.where(thin, torch.maximum((hd * hd / (2 * DESING) + 0.5 * DESING).clamp_max(DESING), hd.abs()), hd)
        u, v = torch.where(closed, z, hu / den), torch.where(closed, z, hv / den)
        E = torch.where(self.land, torch.full_like(h, DRY), torch.where(dry, CUTOFF - self.Hm, e))
        flag = (E == DRY)
        J, I = slice(2, self.ny + 2), slice(2, self.nx + 2)
        f, dx = self.f, self.dx
        T, F = _axis_fluxes(E[..., J, :], u[..., J, :], v[..., J, :], self.W[J], self.Ea[J], flag[..., J, :],
                            self.fx, self.ax, -1.0, f[J], dx)
        y = lambda x: x[..., :, I].transpose(-1, -2)  # noqa: E731
        S, Gf = _axis_fluxes(y(E), y(v), y(u), y(self.S), y(self.N), y(flag), self.fy, self.ay, 1.0,
                             f.transpose(0, 1), dx)
        S = S.transpose(-1, -2)
        Gf = [x.transpose(-1, -2) for x in (Gf[0], Gf[2], Gf[1])]
        L = [-(a[..., 1:] - a[..., :-1]) / dx - (b[..., 1:, :] - b[..., :-1, :]) / dx for a, b in zip(F, Gf)]
        ec, uc, vc, Hc = E[..., J, I], u[..., J, I], v[..., J, I], self.Hc[J, I]
        h = ec + Hc
        hu, hv = (torch.where(h > CUTOFF, x * h, torch.zeros_like(h)) for x in (uc, vc))
        on = (h >= CUTOFF) & ~flag[..., J, I]
        sx = self.X + f[J] * hv + GRAV * h * (self.Ea - self.W)[J, I] / dx
        sy = self.Y - f[J] * hu + GRAV * h * (self.N - self.S)[J, I] / dx
        L[1] = L[1] + torch.where(on, sx, torch.zeros_like(h))
        L[2] = L[2] + torch.where(on, sy, torch.zeros_like(h))
        new = [a + dt * b for a, b in zip((ec, hu, hv), L)]
        if qn is not None:
            new = [0.5 * (q[..., J, I] + a) for q, a in zip(qn, new)]
        gone = new[0] + Hc <= CUTOFF
        new = [torch.where(gone, CUTOFF - Hc, new[0])] + [torch.where(gone, torch.zeros_like(h), a) for a in new[1:]]
        return [torch.nn.functional.pad(a, (2, 2, 2, 2)) for a in new]

    def step(self, e, hu, hv, dt):
        a = self.stage(e, hu, hv, dt)
        return tuple(self.stage(*a, dt, (e, hu, hv)))

    def finish(self, q, q0):
        """The padded state as a step leaves it: the ghost cells that image
        an interior cell follow it, the others keep what they held."""
        J, I = slice(2, self.ny + 2), slice(2, self.nx + 2)
        A, B = (slice(None) if self.ns else J), (slice(None) if self.ew else I)
        out = [b.clone() for b in q0]
        for a, n in zip(out, q):
            a[..., A, B] = n[..., self.rows, :][..., :, self.cols][..., A, B]
        return out

    def exchange(self, q):
        """Periodic ghost rows and columns, over their whole length."""
        for a in q:
            if self.ns:
                a.copy_(a[..., self.rows, :])
            if self.ew:
                a.copy_(a[..., :, self.cols])
        return q

    def start(self, q):
        """The initial state as the constructors take it."""
        q = [a.double().clone() for a in q]
        q[0] = torch.maximum(q[0], -torch.where(self.land, torch.full_like(self.Hm, LAND), self.Hm))
        return q


def _wind_fields(case, seed, nx, ny):
    X, Y = (torch.from_numpy(a).cuda().double() for a in _wind(case, seed))
    if X.numel() == 1:
        return float(X), float(Y)

    def axis(n, w):
        x = (torch.arange(2, n + 2, device="cuda", dtype=F64) + 0.5) / n * w - 0.5
        k = x.floor()
        i = k.long()
        return i.clamp(0, w - 1), (i + 1).clamp(0, w - 1), x - k
    r0, r1, b = axis(ny, X.shape[0])
    c0, c1, a = axis(nx, X.shape[1])
    b = b[:, None]
    return [(1 - b) * ((1 - a) * F[r0][:, c0] + a * F[r0][:, c1]) + b * ((1 - a) * F[r1][:, c0] + a * F[r1][:, c1])
            for F in (X, Y)]


def _normals(n, key, counter, first, members):
    """(members, n) normal numbers of the counter-based generator Philox4x32-10
    (Salmon, Moraes, Dror, Shaw: Parallel random numbers, SC'11) and
    Box-Muller, of the members from ``first`` on."""
    nt = (n + 3) // 4
    m32 = np.uint64(0xFFFFFFFF)
    who = np.arange(first, first + members, dtype=np.uint64)[:, None]
    c = [np.ascontiguousarray(np.broadcast_to(x, (members, nt))) for x in
         (np.arange(nt, dtype=np.uint64)[None], np.uint64(counter), np.uint64(0), who)]
    k = [np.uint64(key & 0xFFFFFFFF), np.uint64(key >> 32)]
    for rnd in range(10):
        if rnd:
            k = [(k[0] + np.uint64(0x9E3779B9)) & m32, (k[1] + np.uint64(0xBB67AE85)) & m32]
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ k[0], b & m32, (a >> np.uint64(32)) ^ c[3] ^ k[1], a & m32]
    u = [torch.from_numpy(((x >> np.uint64(9)).astype(np.float64) + 0.5) * 2.0 ** -23).cuda() for x in c]
    r = [torch.sqrt(-2 * torch.log(u[i])) for i in (0, 2)]
    w = [2 * math.pi * u[i] for i in (1, 3)]
    z = torch.stack([r[0] * torch.cos(w[0]), r[0] * torch.sin(w[0]), r[1] * torch.cos(w[1]), r[1] * torch.sin(w[1])], -1)
    return z.reshape(members, -1)[:, :n]


def _catmull_rom(n, factor):
    """(n + 2, n / factor + 4) weights of the cubic interpolation of a coarse
    axis at the fine cells -1 .. n, both with two ghost cells in front."""
    cn = n // factor
    x = (torch.arange(-1, n + 1, dtype=F64) + 0.5) / factor + 1.5
    c = x.floor().long()
    c = torch.where(c > cn + 1, c - 1, c)
    t = (x - c)[:, None]
    w = torch.cat([-t + 2 * t ** 2 - t ** 3, 2 - 5 * t ** 2 + 3 * t ** 3, t + 4 * t ** 2 - 3 * t ** 3, -t ** 2 + t ** 3], 1) / 2
    W = torch.zeros(n + 2, cn + 4, dtype=F64)
    for k in range(4):
        W.scatter_add_(1, (c + k - 1).clamp(0, cn + 3)[:, None], w[:, k:k + 1])
    return W.cuda()


def _model_error(sch, factor, key, counter, first, q):
    """Adds a random eta of the SOAR covariance and the transports in balance
    with it to the members from ``first`` on."""
    members = q[0].shape[0]
    nx, ny, dx = sch.nx, sch.ny, sch.dx
    cx, cy, cd = nx // factor, ny // factor, dx * factor
    gx, gy = (0 if p else 4 for p in (sch.ew, sch.ns))
    xi = _normals((cx + 2 * gx) * (cy + 2 * gy), key, counter, first, members).view(members, cy + 2 * gy, cx + 2 * gx)
    L = 0.75 * cd
    ax, ay = torch.arange(cx + 4, device="cuda"), torch.arange(cy + 4, device="cuda")
    C = 0.0
    for oy in range(-2, 3):
        for ox in range(-2, 3):
            r = math.hypot(ox, oy) * cd / L
            i = (ax - 2 + ox) % cx if sch.ew else ax + 2 + ox
            j = (ay - 2 + oy) % cy if sch.ns else ay + 2 + oy
            C = C + float(np.float32(Q0)) * (1 + r) * math.exp(-r) * xi[:, j][:, :, i]
    if factor > 1:
        wx, wy = _catmull_rom(nx, factor), _catmull_rom(ny, factor)
        d = torch.matmul(torch.matmul(wy, C.contiguous()), wx.t().contiguous())
    else:
        d = C[:, 1:ny + 3, 1:nx + 3]
    J, I = slice(2, ny + 2), slice(2, nx + 2)
    dc = d[:, 1:-1, 1:-1]
    h = dc + sch.Hc[J, I] + (q[0][..., J, I] if factor == 1 else 0.0)
    k = GRAV / sch.f[J] / (2 * dx) * h
    out = [a.clone() for a in q]
    out[0][..., J, I] += dc
    out[1][..., J, I] -= k * (d[:, 2:, 1:-1] - d[:, :-2, 1:-1])
    out[2][..., J, I] += k * (d[:, 1:-1, 2:] - d[:, 1:-1, :-2])
    return out


def _drift(sch, P, q, dt):
    """Drifters (members, n, 2) moved by the interpolated velocity; the cell
    is taken one to the north-east, as the scheme's drifters do."""
    c, f = torch.ceil(P / sch.dx) + 2, P / sch.dx - torch.floor(P / sch.dx)
    lo = torch.where(f < 0.5, c - 1, c).long()
    w = torch.where(f < 0.5, f + 0.5, f - 0.5)
    m = torch.arange(P.shape[0], device="cuda")[:, None]
    vel = []
    top = torch.tensor([sch.nx + 3, sch.ny + 3], device="cuda")
    for x in q[1:]:
        s = 0.0
        for b in (0, 1):
            for a in (0, 1):
                i, j = (torch.minimum(lo + torch.tensor([a, b], device="cuda"), top)[..., k] for k in (0, 1))
                wt = (w[..., 0] if a else 1 - w[..., 0]) * (w[..., 1] if b else 1 - w[..., 1])
                s = s + wt * x[m, j, i] / (sch.Hm[j, i] + q[0][m, j, i])
        vel.append(s)
    P = P + dt * torch.stack(vel, -1)
    size = torch.tensor([sch.nx * sch.dx, sch.ny * sch.dx], device="cuda", dtype=F64)
    on = torch.tensor([sch.ew, sch.ns], device="cuda")
    P = torch.where(on & (P < 0), P + size, P)
    return torch.where(on & (P > size), P - size, P)


def _exact_ens(case, seed):
    nx, ny, dx, members = case["nx"], case["ny"], _dx(case), case["members"]
    eta, hu, hv, Hi = _domain(case, seed, members, nx, ny, dx)
    sch, dt = _Scheme(case, nx, ny, dx, Hi), _dt(Hi, dx)
    key, num = 0, case.get("drifters") or 0
    if case.get("noise"):
        rs = np.random.RandomState(seed & 0xFFFFFF)
        key = int(rs.randint(0, 2 ** 31)) | (int(rs.randint(0, 2 ** 31)) << 31)
    P = torch.zeros((members, num + 1, 2), dtype=F64, device="cuda")
    if num:
        rows = max(1, round(math.sqrt(num)))
        cols = -(-num // rows)
        k = torch.arange(num, device="cuda")
        P[:, :num, 0] = (((k % cols).double() + 0.5) * nx * dx / cols).float().double()
        P[:, :num, 1] = ((torch.div(k, cols, rounding_mode="floor").double() + 0.5) * ny * dx / rows).float().double()
    out = torch.empty((members, 3, ny + 4, nx + 4), dtype=F64, device="cuda")
    # a few members at a time: the scheme's temporaries are many planes each
    for a in range(0, members, 16):
        b = min(members, a + 16)
        q, p = sch.exchange(sch.start((eta[a:b], hu[a:b], hv[a:b]))), P[a:b]
        for n in range(case["steps"]):
            q = sch.finish(sch.step(*q, dt), q)
            if case.get("noise"):
                q = _model_error(sch, case["noise"], key, n, a, q)
                q = sch.exchange(q)
            if num:
                p = _drift(sch, p, q, dt)
        out[a:b] = torch.stack(q, 1)
        P[a:b] = p
    got = {"state": out.reshape(-1)}
    if num:
        c = (torch.floor(P[:, :num].float().double() / dx) + 2).long()
        m = torch.arange(members, device="cuda")[:, None]
        got["observed"] = torch.stack([out[m, k, c[..., 1], c[..., 0]] for k in (1, 2)], -1)
        got["drifters"] = P[:, :num]
    return got



def _exact_step(case, seed):
    nx, ny, dx = case["nx"], case["ny"], _dx(case)
    eta, hu, hv, Hi = _domain(case, seed, 1, nx, ny, dx)
    sch = _Scheme(case, nx, ny, dx, Hi, *_wind_fields(case, seed, nx, ny))
    q, dt = sch.start([a[0] for a in (eta, hu, hv)]), _dt(Hi, dx)
    if not case.get("cfl"):
        for _ in range(case["steps"]):
            q = sch.finish(sch.step(*q, dt), q)
        return dict(zip(("eta", "hu", "hv"), q))
    q, t, end = sch.exchange(q), 0.0, case["steps"] * dt * 0.97
    J, I = slice(2, ny + 2), slice(2, nx + 2)
    while t < end:
        h = (q[0] + sch.Hm)[J, I]
        wet = ~sch.land[J, I] & (h > 0)
        c = torch.sqrt(GRAV * h.clamp_min(0.0))
        v = torch.maximum((q[1][J, I] / h).abs() + c, (q[2][J, I] / h).abs() + c)
        local = min(0.6 * 0.25 * dx / float(v[wet].max()), end - t)
        q = sch.finish(sch.step(*q, local), q)
        t += local
    return dict(zip(("eta", "hu", "hv"), q))


def _exact_gradient(sch, q0, dt, steps, nx, ny, dx, seed):
    """Misfit, final state and gradient by autograd."""
    leaf = [a.requires_grad_(True) for a in q0]
    q = tuple(leaf)
    for _ in range(steps):
        q = checkpoint(sch.step, *q, dt, use_reentrant=False)
    ox, oy, y = _points(nx, ny, dx, seed, 64)
    fx, fy = (torch.from_numpy(a / dx + 1.5).cuda() for a in (ox, oy))
    i, j = fx.floor().long(), fy.floor().long()
    a, b = fx - i, fy - j
    e = q[0]
    got = (1 - b) * ((1 - a) * e[j, i] + a * e[j, i + 1]) + b * ((1 - a) * e[j + 1, i] + a * e[j + 1, i + 1])
    J = 0.5 * ((got - torch.from_numpy(y).cuda().double()) ** 2).sum()
    grad = torch.autograd.grad(J, leaf)
    with torch.no_grad():
        return J.detach(), sch.finish([x.detach() for x in q], [x.detach() for x in leaf]), list(grad)


def _exact_letkf(case, seed):
    """Every group of buoys in turn: the local transform of each buoy's box,
    blended with its weights (R the unit matrix, no inflation)."""
    nx, ny, dx, N, r = case["nx"], case["ny"], _dx(case), case["members"], _letkf_r(case)
    eta, hu, hv, Hi = _domain(case, seed, N, nx, ny, dx)
    sch = _Scheme(case, nx, ny, dx, Hi)
    q = sch.exchange(sch.start((eta, hu, hv)))
    full = torch.stack(q, 1)                                     # (N, 3, ny + 4, nx + 4)
    X = full[:, :, 2:-2, 2:-2].clone()
    obs = _buoys(case, seed)
    R = math.ceil(1.5 * r)
    o = np.arange(-R, R + 1)
    dist = np.hypot(o[None, :], o[:, None])
    z = np.minimum.reduce([np.hypot(o[None, :] + a * nx, o[:, None] + b * ny) for a in (0, -1, 1) for b in (0, -1, 1)]) / r
    with np.errstate(divide="ignore", invalid="ignore"):
        w = np.where(z < 1, 1 - 5 / 3 * z ** 2 + 5 / 8 * z ** 3 + z ** 4 / 2 - z ** 5 / 4,
                     4 - 5 * z + 5 / 3 * z ** 2 + 5 / 8 * z ** 3 - z ** 4 / 2 + z ** 5 / 12 - 2 / (3 * z))
    w = np.where((dist <= 1.5 * r) & (z < 2), np.minimum(1.0, w), 0.0)
    jj, ii = np.nonzero(w)
    wt = torch.from_numpy(w[jj, ii]).cuda()
    # groups whose buoys are 3 r cells apart: the later of the closest pair
    # moves on while there is a closer one
    lx, ly = nx * dx, ny * dx
    d = np.abs(obs[:, None, :2] - obs[None, :, :2])
    d = np.hypot(np.where(d[..., 0] > lx / 2, lx - d[..., 0], d[..., 0]), np.where(d[..., 1] > ly / 2, ly - d[..., 1], d[..., 1]))
    np.fill_diagonal(d, math.hypot(lx, ly))
    groups, k = [list(range(len(obs)))], 0
    while k < len(groups):
        while len(groups[k]) > 1:
            sub = d[np.ix_(groups[k], groups[k])]
            at = int(sub.argmin())
            if sub.flat[at] >= 3 * r * dx:
                break
            if len(groups) == k + 1:
                groups.append([])
            groups[k + 1].append(groups[k].pop(at % len(groups[k])))
        k += 1
    one = torch.eye(N, dtype=F64, device="cuda")
    for group in groups:
        mean = X.mean(0)
        W, add = torch.zeros((ny, nx), dtype=F64, device="cuda"), torch.zeros_like(X)
        for b in group:
            cx, cy = (int(math.floor(obs[b, k] / dx)) for k in (0, 1))
            hx = X[:, 1:, cy, cx]
            hp = (hx - hx.mean(0)).t()                           # (2, N)
            D = torch.from_numpy(obs[b, 2:]).cuda() - hx.mean(0)
            A = (N - 1) * one + hp.t().contiguous() @ hp
            lam, V = torch.linalg.eigh(A)
            P = (V * torch.sqrt((N - 1) / lam)) @ V.t().contiguous()
            P = P + torch.linalg.solve(A, hp.t().contiguous() @ D)[:, None]
            j = torch.from_numpy((int(np.round(obs[b, 1] / dx)) - R + jj) % ny).cuda()
            i = torch.from_numpy((int(np.round(obs[b, 0] / dx)) - R + ii) % nx).cuda()
            loc, m = X[:, :, j, i], mean[:, j, i]
            new = (P.t().contiguous() @ (loc - m).reshape(N, -1)).reshape(loc.shape) + m
            W[j, i] += wt
            add[:, :, j, i] += new * wt
        X = (1 - W / W.clamp_min(1.0)) * X + add
    full[:, :, 2:-2, 2:-2] = X
    return {"state": torch.stack(sch.exchange(list(full.unbind(1))), 1).reshape(-1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "ens":
        return _exact_ens(case, seed)
    if kind == "letkf":
        return _exact_letkf(case, seed)
    dx = _dx(case)
    if kind == "adj":
        nx, ny = case["nx"], case["ny"]
        eta, hu, hv, Hi = _domain(case, seed, 1, nx, ny, dx)
        sch = _Scheme(case, nx, ny, dx, Hi)
        q = sch.start([a[0] for a in (eta, hu, hv)])
        J, state, grad = _exact_gradient(sch, q, _dt(Hi, dx), case["steps"], nx, ny, dx, seed)
        return {"J": J, "state": state, "grad": grad}
    J, state, grad = 0.0, [], []
    for k, (nx, ny) in enumerate(_sides(case)):
        eta, hu, hv, Hi = _domain(case, seed * 31 + k, 1, nx, ny, dx)
        sch = _Scheme(case, nx, ny, dx, Hi)
        q = sch.start([a[0] for a in (eta, hu, hv)])
        one = _exact_gradient(sch, q, _dt(Hi, dx), case["steps"], nx, ny, dx, seed + k)
        J = J + one[0]
        state += [a.reshape(-1) for a in one[1]]
        grad += [a.reshape(-1) for a in one[2]]
    return {"J": J, "state": torch.cat(state), "grad": torch.cat(grad)}
