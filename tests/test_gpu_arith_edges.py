"""The kernels' FP64 quotient on the device where it lies next to the middle of
two doubles: dividends and divisors within 63 units of a power of two on either
side, among them a power of two over a divisor whose mantissa is all ones."""
import numpy as np
import pytest

from cffc_amd import euler2d

pytestmark = pytest.mark.gpu


def test_quotients_next_to_a_midpoint():
    rng = np.random.default_rng(5)
    k = np.arange(64)
    m = np.concatenate([1.0 + k * 2.0**-52, 2.0 - (k + 1) * 2.0**-52])
    a, b = (q.ravel() for q in np.meshgrid(m, m))
    a, b = np.tile(a, 8), np.tile(b, 8)
    a = np.ldexp(a, rng.integers(-300, 300, a.size)) * rng.choice([-1.0, 1.0], a.size)
    b = np.ldexp(b, rng.integers(-300, 300, b.size)) * rng.choice([-1.0, 1.0], b.size)
    o = euler2d.check_arith(a, b)
    assert np.array_equal(np.ascontiguousarray(o[:, 0]).view(np.uint64), (a / b).view(np.uint64))
