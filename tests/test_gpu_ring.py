"""The faithful boundary phase in one launch against the oracle's passes
(lid_driven_cavity/src/lbm.cpp:233-301, sphere/src/lbm.cpp:277-356), bit for bit:
where a source lies in another pass's ghost plane, deeper than the first ghost
layer, or across the whole domain, and on both sides of the rule that puts
usrbc into the same launch."""
import numpy as np
import pytest

from oracle.oracle import FAITHFUL, LDC, SPHERE, Oracle

pytestmark = pytest.mark.gpu


def steps_equal(case, n, tau):
    from imexlb_amd import LBM
    o = Oracle(case, *n, tau0=tau, u0=0.1, mode=FAITHFUL, lid_u=0.1)
    o.Initialize()
    g = LBM(*n, tau, u0=0.1, case=case, mode=FAITHFUL, engine="fused", lid_u=0.1)
    g.Initialize()
    for k in (1, 2, 9):  # odd and even: each of the two rings ends up last
        o.run(k)
        g.step(k)
        for a, b in zip(o.moments(), g.moments()):
            assert np.array_equal(a, b), (case, n, k)
    o.Collision()
    assert np.array_equal(o.get_f(), g.get_f())


@pytest.mark.parametrize("n", [(2, 2, 2), (2, 2, 3), (3, 3, 3), (4, 4, 4), (2, 5, 9), (65, 3, 4), (3, 66, 5), (17, 4, 67)])
def test_cavity_ring(n):
    steps_equal(LDC, n, 0.2)


# lo >= 2 first holds at nx = 25 (box 2..4: extents from 7); at nx = 72 the box
# is 6..10 (extents from 13), at nx = 66 also radius 2
@pytest.mark.parametrize("n", [(24, 9, 9), (25, 7, 8), (25, 6, 8), (25, 8, 6), (72, 13, 13), (72, 13, 12), (66, 14, 15),
                               (4, 2, 2), (2, 3, 2)])
def test_sphere_ring(n):
    steps_equal(SPHERE, n, 0.08)
