"""Speeds and populations at the ends of FP64's range: what the collision's reciprocal
division (fused.h div_by) gives where it applies, and IEEE's elsewhere."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 1e153: u^2 is finite; 1e154 and more: it overflows, and feq with it, while the
# populations, which the choice of the division looks at, are of size one
@pytest.mark.parametrize("u0", [1e100, 1e153, 1e154, 1e160, 1e300])
def test_inlet_speeds_beyond_the_populations(u0):
    from imexlb_amd import LBM
    n = (72, 20, 20)
    print(f"[case] inlet speed {u0}", flush=True)
    f = np.random.default_rng(5).uniform(0.5, 1.5, (27, n[2], n[1], n[0]))
    out = []
    for am in (2, -1):
        with LBM(*n, 0.024, u0=u0, case="sphere", mode="faithful", addr_mode=am) as g:
            g.Initialize()
            g.set_f(f)
            g.step(1)
            out.append([g.get_f()] + g.moments())
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
