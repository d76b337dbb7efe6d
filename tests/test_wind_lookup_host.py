"""The bracketing wind samples of a model time: the same as a binary search over
the sample times in float64, whatever sequence and type holds them."""

from types import SimpleNamespace

import numpy as np
import pytest

from SWESimulators import Simulator

TIMES = [0.0, 3600.1, 7200.2, 10800.3]


@pytest.mark.parametrize("hold", [list, tuple, lambda t: np.array(t), lambda t: np.array(t, np.float32),
                                  lambda t: np.array(t).astype(np.int64), lambda t: [np.float32(x) for x in t]])
@pytest.mark.parametrize("kind", [float, np.float64])
def test_bracketing_samples(hold, kind):
    ts = hold(TIMES)
    at = sorted({x for t in ts for x in (float(t), np.nextafter(float(t), -1e9), np.nextafter(float(t), 1e9),
                                         float(t) + 5e-5, float(t) + 900.0)} | {-1.0, 2e4})
    for t in at:
        sim = SimpleNamespace(wind_stress=SimpleNamespace(t=ts), t=kind(t))
        k = int(np.searchsorted(np.asarray(ts, np.float64), t))
        i0, i1 = max(0, k - 1), min(len(ts) - 1, k)
        got = Simulator.Simulator.wind_stress_interpolation(sim)
        assert got[:2] == (i0, i1), (t, got)
        assert 0.0 <= got[2] <= 1.0
