"""Planes whose tiles are smaller than a wavefront (one or a few 128-byte lines per
population, kernels.h tile_geom): the same populations and moments as arrays, bit
for bit, on planes that end inside a line, a tile and a wavefront."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANES = [(8, 8, 5), (13, 5, 6), (9, 8, 4), (10, 13, 5), (12, 12, 4), (20, 10, 3), (20, 20, 3), (23, 23, 3)]


def state(n, steps, addr_mode, shape=None, **kw):
    from imexlb_amd import LBM
    with LBM(*n, 0.06, u0=0.05, addr_mode=addr_mode, **kw) as g:
        if shape:
            g.set_launch(*shape)
        g.Initialize()
        g.step(steps, 3)
        return [g.get_f()] + g.moments()


@pytest.mark.parametrize("n", PLANES)
@pytest.mark.parametrize("case,mode,dtype,storage", [
    ("tgv", "faithful", "f64", "pull"), ("tgv", "faithful", "f64", "aa"), ("tgv", "faithful", "f32", "aa"),
    ("cavity", "config", "f64", "aa"), ("cavity", "config", "f32", "pull"), ("cavity", "faithful", "f64", "pull")])
def test_tiles_of_a_few_lines_equal_arrays(n, case, mode, dtype, storage):
    print(f"[case] small tiles {case} {mode} {n} {dtype} {storage}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, storage=storage)
    for steps in (4, 5):
        want = state(n, steps, 2, **kw)
        for shape in (None, (256, 2, 1, 1)):
            for a, b in zip(want, state(n, steps, -1, shape, **kw)):
                assert np.array_equal(a, b), (steps, shape)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_channel_in_tiles_of_a_few_lines(dtype):
    n = (25, 9, 9)
    kw = dict(case="sphere", mode="config", sphere=(8.0, 4.0, 4.0, 2.2), dtype=dtype)
    for a, b in zip(state(n, 5, 2, **kw), state(n, 5, -1, **kw)):
        assert np.array_equal(a, b)
