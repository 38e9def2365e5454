"""x^(-1/4) as the 1D steps take it: from single-precision seeds.

The seed q is a single-precision number, so q^2 is exact; q^4 is rounded once (2^-53,
a quarter of which reaches the result), the series leaves 7.5 d^3 for a seed error d of
2^-22.5 (2^-64.6), and the result is rounded once: below 0.5 + 0.25 + 0.01 units in the
last place."""
import math
import random

import mpmath
import pytest

from geliosphere_amd import engine as E

pytestmark = pytest.mark.gpu


def ulps(y, ref):
    """Against the exact value, not its rounding."""
    return float(abs(mpmath.mpf(y) - ref)) / math.ulp(float(ref))


def test_fourth_root_from_single_precision_seeds(engine):
    mpmath.mp.dps = 50
    rng = random.Random(17)
    xs = [10.0 ** rng.uniform(-30, 36) for _ in range(4000)]
    xs += [1.0 + 15.0 * rng.random() for _ in range(4000)]                 # a period of the mantissa
    xs += [(2 * 2.2e-4 * dt * 0.938272) ** 2 * (1.0 + 10.0 ** rng.uniform(-6, 5))   # alpha^2 E^2
           for dt in (50.0, 500.0) for _ in range(2000)]
    xs += [1.0, 2.0, 4.0, 16.0, 1e-30, 1e36, float.fromhex("0x1.fffffffffffffp+0"), float.fromhex("0x1.0000000000001p+0")]
    ref = [mpmath.mpf(x) ** mpmath.mpf(-0.25) for x in xs]
    mid = max(ulps(a, r) for a, r in zip(engine.debug_math(E.DBG_RSQRT4_MID, xs), ref))
    both = max(ulps(a, r) for a, r in zip(engine.debug_math(E.DBG_RSQRT4, xs), ref))
    print("worst error in units of the last place: single-precision seeds %.3f, double %.3f" % (mid, both))
    assert mid <= 0.77
    assert mid <= both   # no less accurate than the double-precision seeds
