"""The lane polynomials and the update's products at the limits a block has to meet: |d| measured against a r =
a / (1 + a dt0) (sg2_abar_rate), which for a fast pole lies far beyond what a limit on a d would admit."""
import math

import numpy as np
import pytest

from oracle import oracle as orc

L = orc.lib()


@pytest.mark.parametrize("a_lo,a_hi", [(0.01, 1.0), (1.0, 16.0), (16.0, 400.0)])
def test_polynomials_at_the_limit_of_the_rate(a_lo, a_hi):
    """A_bar as a cubic for a r |d| up to 2^-7 and its products with cos / sin as quadratics for (2.3 a r + |f|) |d| up to
    2^-7.5, against float64.  Tolerances: the remainders (2^-27, 3e-8), three fp32 roundings of the value (4e-7 relative
    covers them) and one each of the constant 2 r - 1 and its products, whose terms are of order 1 (1.5e-7, 2e-7)."""
    r = np.random.RandomState(11)
    for _ in range(3000):
        dt0 = float(np.float32(r.uniform(0.02, 3.0)))
        ae, ao = (float(np.float32(np.exp(r.uniform(np.log(a_lo), np.log(a_hi))))) for _ in range(2))
        f = float(np.float32(r.uniform(-1.0, 1.0)))
        rate = max(a / (1.0 + a * dt0) for a in (ae, ao))
        sign = r.choice((-1.0, 1.0))
        d = float(np.float32(sign * r.uniform(0.9, 1.0) * 2.0 ** -7 / rate))
        for a in (ae, ao):
            dt = dt0 + d
            exact = (1.0 - a * dt) / (1.0 + a * dt)
            assert abs(L.orc_abar_poly(dt0, a, d) - exact) <= 4e-7 * abs(exact) + 1.5e-7, (dt0, a, d)
        d = float(np.float32(sign * r.uniform(0.9, 1.0) * 2.0 ** -7.5 / (2.3 * rate + abs(f))))
        dt = dt0 + d
        A = [(1.0 - a * dt) / (1.0 + a * dt) for a in (ae, ao)]
        want = (A[0] * math.cos(f * dt), -A[0] * math.sin(f * dt), A[1] * math.cos(f * dt), A[1] * math.sin(f * dt))
        for which in range(4):
            got = L.orc_pair_product(dt0, ae, ao, f, d, which)
            assert abs(got - want[which]) <= 4e-7 * abs(want[which]) + 2e-7, (dt0, ae, ao, f, d, which)
