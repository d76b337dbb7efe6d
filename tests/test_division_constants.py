"""The host's choice of constants for the substep kernels' division by the cell
sizes and 2g, RN(n high + RN(n low)): the pair is exact, checked here with NumPy,
also for divisors for which the correctly rounded low part alone is not."""

import ctypes

import numpy as np
import pytest

from SWESimulators import _gocean as G

F = np.float32
# divisors whose rounded low part gives a wrong last place for some n
HARD = [1000.0 / 3.0, float.fromhex("0x1.c3f856p+8"), float.fromhex("0x1.d6be26p+9"),
        float.fromhex("0x1.8f22aep+4"), float.fromhex("0x1.e22acep+6"), float.fromhex("0x1.749b7ep-2")]
PLAIN = [2 * 9.81, 200.0, 77.7, 4.0, 800.0]


def _constants(d):
    hi, lo = ctypes.c_float(), ctypes.c_float()
    ok = G.load().gocean_division_constants(float(F(d)), ctypes.byref(hi), ctypes.byref(lo))
    return ok, F(hi.value), F(lo.value)


def _quotients(n, hi, lo):
    """RN(n hi + RN(n lo)): the product of two floats and its sum with the float
    n lo fit the 64 bits of a long double, so one rounding to float is left."""
    return (n.astype(np.longdouble) * np.longdouble(hi) + (n * lo).astype(np.longdouble)).astype(F)


@pytest.mark.parametrize("d", HARD + PLAIN)
def test_fast_division_is_available_and_exact(d):
    ok, hi, lo = _constants(d)
    assert ok == 1, d
    assert hi == F(1.0) / F(d)
    for k in range(8):                         # every significand of n in [1, 2)
        n = (np.arange(k << 20, (k + 1) << 20, dtype=np.uint32) | np.uint32(0x3F800000)).view(F)
        assert np.array_equal(_quotients(n, hi, lo), n / F(d))


@pytest.mark.parametrize("d", [300.0, 2 * 9.81, 1000.0 / 3.0])
def test_fast_division_of_tiny_values(d):
    """Exact while n low is normal; below, within one unit in the last place:
    n low is then off by at most 2^-150, half the smallest spacing of floats."""
    ok, hi, lo = _constants(d)
    assert ok == 1
    rng = np.random.default_rng(1)
    limit = 2.0 ** -126 / abs(float(lo))       # of |n|
    sig = (1 + rng.random(200_000)).astype(F)
    for e in range(-125, -60, 4):
        n = sig * F(2.0 ** e)
        with np.errstate(under="ignore"):
            got, want = _quotients(n, hi, lo), n / F(d)
        if 2.0 ** e >= limit:
            assert np.array_equal(got, want), e
        else:
            assert np.all(np.abs(got.view(np.int32) - want.view(np.int32)) <= 1), e


@pytest.mark.parametrize("d", [0.0, -2.0, float("nan"), float("inf"), 1e-45, 3e38])
def test_divisors_without_a_normal_reciprocal(d):
    assert _constants(d)[0] == 0
    assert G.load().gocean_division_constants(1.0, None, None) < 0
