"""GPU: the reciprocal root and e^-x of the FP64 kernels (rsqrt_nr, exp_neg64)
against the host's 80-bit long double."""
import numpy as np
import pytest

from beep3_amd._lib import dp, lib
from beep3_amd.device import Device

pytestmark = pytest.mark.gpu

N = 4_000_000
LD = np.longdouble
needs_80_bits = pytest.mark.skipif(np.finfo(LD).nmant < 63, reason="needs an 80-bit long double")


def run(which, x):
    d = Device(0)
    x = np.ascontiguousarray(x, dtype=np.float64)
    y = np.empty_like(x)
    d._check(lib().beep_hip_selftest_math(d._h, which, len(x), x.ctypes.data_as(dp), y.ctypes.data_as(dp)))
    d.close()
    return y


def errors(y, exact):
    """Largest and root mean square relative error in units of 2^-53."""
    e = np.abs((y.astype(LD) - exact) / exact).astype(np.float64) * 2.0 ** 53
    return float(e.max()), float(np.sqrt(np.mean(e * e)))


@needs_80_bits
@pytest.mark.parametrize("lo,hi", [(0.25, 4.0), (1e-30, 1e-8), (1e8, 1e30), (1e-290, 1e-280), (1e280, 1e290)])
def test_reciprocal_root(lo, hi):
    """The last rounding is at most one unit, the rounding of v y adds half
    of one, the series less than 0.01."""
    x = np.exp(np.random.default_rng(1).uniform(np.log(lo), np.log(hi), N))
    worst, rms = errors(run(0, x), 1 / np.sqrt(x.astype(LD)))
    print("rsqrt", lo, hi, worst, rms)
    assert worst < 1.51 and rms < 0.5


@needs_80_bits
@pytest.mark.parametrize("hi", [0.4, 30.0, 700.0])
def test_exponential(hi):
    """The last rounding is at most one unit, the one before it, of a number
    up to 0.42 apart from 1, at most 0.6 of one, that of the reduced argument
    a quarter, the polynomial less than 0.06."""
    x = np.random.default_rng(2).uniform(0.0, hi, N)
    worst, rms = errors(run(1, x), np.exp(-x.astype(LD)))
    print("exp", hi, worst, rms)
    assert worst < 1.91 and rms < 0.5


def test_ends():
    assert np.array_equal(run(1, [0.0, 746.0, 750.0, 1e4, 1e300, np.inf]), [1.0, 0.0, 0.0, 0.0, 0.0, 0.0])
    tail = np.linspace(700.0, 745.0, 1000)  # down to the smallest number, 2^-1074
    assert np.all(np.abs(run(1, tail) - np.exp(-tail)) <= 2.0 ** -1073 + 4e-16 * np.exp(-tail))
    p = 4.0 ** np.arange(-500, 500)
    assert np.array_equal(run(0, p), 2.0 ** -np.arange(-500.0, 500.0))
