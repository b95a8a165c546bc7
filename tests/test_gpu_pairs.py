"""Two adjacent cells per thread (cells_per_thread 3) over arrays, where its kernel
runs: an explicit addr_mode selects them, and imexlb_get_info says that the kernel is
in effect, so that a change of the default layout cannot empty these tests."""
import numpy as np
import pytest

from oracle.oracle import FAITHFUL, TGV, Oracle

pytestmark = pytest.mark.gpu

# rows of one pair, of part of a wavefront, of whole and of several wavefronts, with
# row ends inside and at the end of a wavefront and of a workgroup
EXTENTS = [(2, 3, 2), (4, 2, 3), (6, 5, 3), (64, 3, 2), (66, 5, 3), (130, 3, 3), (256, 2, 2), (128, 40, 3)]
SHAPES = [(64, 3, 0, 0), (128, 3, 1, 1), (256, 3, 1, 1), (512, 3, 1, 0)]


def tau(n):
    return 0.05 * n[0] / 100.0 / (1.0 / 3.0) / 2 / 3.1415926


@pytest.mark.parametrize("n", EXTENTS)
@pytest.mark.parametrize("storage", ["pull", "aa"])
def test_pairs_equal_the_oracle(n, storage):
    from imexlb_amd import LBM
    print(f"[case] pairs {n} {storage}", flush=True)
    o = Oracle(TGV, *n, tau0=tau(n), u0=0.05, mode=FAITHFUL)
    o.Initialize()
    o.run(5)
    want = o.moments()
    o.Collision()
    f = o.get_f()
    for shape in SHAPES:
        with LBM(*n, tau(n), u0=0.05, storage=storage, addr_mode=2) as g:
            g.set_launch(*shape)
            assert g.info()["cells_per_thread"] == 3 and g.info()["addr_mode"] == 2
            g.Initialize()
            g.step(5)
            for a, b in zip(want, g.moments()):
                assert np.array_equal(a, b), shape
            assert np.array_equal(f, g.get_f()), shape


@pytest.mark.parametrize("n", EXTENTS)
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("storage", ["pull", "aa"])
def test_pairs_equal_single_cells(n, dtype, storage):
    from imexlb_amd import LBM
    print(f"[case] pairs {n} {dtype} {storage}", flush=True)
    runs = []
    for shape in [(256, 1, 1, 0)] + SHAPES:
        with LBM(*n, tau(n), u0=0.05, dtype=dtype, storage=storage, addr_mode=2) as g:
            g.set_launch(*shape)
            assert g.info()["cells_per_thread"] == shape[1]
            g.Initialize()
            g.step(5)
            runs.append([g.get_f()] + g.moments())
    for r in runs[1:]:
        for a, b in zip(runs[0], r):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_pairs_after_a_placement_search(dtype):
    """A search and then the pair shape, as a tuned run has it: the same result whichever
    layout the search kept, and pairs in effect if it kept arrays."""
    from imexlb_amd import LBM
    n = (192, 160, 90)
    print(f"[case] pairs after a search {dtype}", flush=True)
    with LBM(*n, 0.05, u0=0.05, dtype=dtype, storage="aa") as g:
        g.Initialize()
        g.step(33)
        want = [g.get_f()] + g.moments()
        g.tune_placement_window(slack_gib=1, step_gib=1 / 4, steps=4)
        g.set_launch(128, 3, 1, 1)
        assert g.info()["cells_per_thread"] == (3 if g.info()["addr_mode"] == 2 else 1)
        g.Initialize()
        g.step(33)
        for a, b in zip(want, [g.get_f()] + g.moments()):
            assert np.array_equal(a, b)
    with LBM(*n, 0.05, u0=0.05, dtype=dtype, storage="aa", addr_mode=2, block=128, cells_per_thread=3) as g:
        assert g.info()["cells_per_thread"] == 3
        g.tune_placement(2, steps=4)
        assert g.info()["cells_per_thread"] == 3
        g.Initialize()
        g.step(33)
        for a, b in zip(want, [g.get_f()] + g.moments()):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("scale", [2.0 ** -1060, 2.0 ** -601, 2.0 ** 401, "mixed"])
@pytest.mark.parametrize("storage", ["pull", "aa"])
def test_scaled_populations_of_planes_below_a_wavefront(scale, storage):
    """test_gpu_division.py's populations far from 1, on a plane that is in arrays by default."""
    from . import test_gpu_division as D
    D.test_scaled_populations(scale, (9, 7, 9), storage)
