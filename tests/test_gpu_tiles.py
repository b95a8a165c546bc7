"""The plane-tile layout (kernels.h LatGeom, tile.h) against the structure of
arrays, which an explicit addr_mode selects and the oracle checks: the same
populations and moments, bit for bit, in every case, storage and launch shape,
on planes that end inside a tile, a workgroup or a wavefront."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (32, 16): one tile of 512 cells; (45, 37), (129, 33): ragged rows and
# tiles; (64, 64), (128, 32): whole tiles; (700, 2) and (2, 300): one and many
# rows per workgroup; (64, 9), (192, 7), (512, 3): rows of one, three and eight
# wavefronts, with rows left over in the last workgroup
PLANES = [(32, 16, 3), (45, 37, 5), (64, 64, 4), (128, 32, 3), (129, 33, 4), (700, 2, 3), (2, 300, 2),
          (64, 9, 4), (192, 7, 3), (512, 3, 2)]
SHAPES = [None, (64, 1, 0, 0), (512, 2, 1, 1), (192, 3, 1, 1)]


def state(n, steps, shape=None, addr_mode=-1, tau=0.06, **kw):
    from imexlb_amd import LBM
    g = LBM(*n, tau, u0=0.05, addr_mode=addr_mode, **kw)
    if shape is not None:
        g.set_launch(*shape)
    g.Initialize()
    g.step(steps, 3)
    f, m = g.get_f(), g.moments()
    info = g.info()
    g.close()
    return f, m, info


def same(a, b, what):
    assert np.array_equal(a[0], b[0]), f"populations: {what}"
    for name, x, y in zip("puvw", a[1], b[1]):
        assert np.array_equal(x, y), f"moment {name}: {what}"


@pytest.mark.parametrize("n", PLANES)
@pytest.mark.parametrize("case,mode", [("tgv", "faithful"), ("cavity", "config")])
@pytest.mark.parametrize("dtype,storage", [("f64", "pull"), ("f64", "aa"), ("f32", "aa"), ("f16", "pull"), ("f16", "aa")])
def test_tiles_equal_arrays(n, case, mode, dtype, storage):
    print(f"[case] tiles {case} {n} {dtype} {storage}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, storage=storage)
    for steps in (6, 7):
        want = state(n, steps, addr_mode=2, **kw)
        for shape in SHAPES:
            got = state(n, steps, shape, **kw)
            same(got, want, f"{steps} steps, launch {shape}")
            assert got[2]["cells_per_thread"] == (2 if shape and shape[1] == 2 else 1)


BOUNDED = [
    ("cavity", "faithful", (24, 30, 5), "f64", None),
    ("cavity", "faithful", (100, 41, 6), "f64", None),
    ("sphere", "faithful", (72, 20, 18), "f64", None),
    ("sphere", "faithful", (130, 37, 40), "f64", None),
    ("sphere", "config", (40, 24, 24), "f64", (12.0, 11.0, 12.0, 4.5)),
    ("sphere", "config", (67, 33, 30), "f16", (20.0, 16.0, 15.0, 5.0)),
    ("sphere", "config", (64, 32, 30), "f32", (20.0, 16.0, 15.0, 12.0)),
]


@pytest.mark.parametrize("case,mode,n,dtype,ball", BOUNDED)
def test_tiles_equal_arrays_at_boundaries(case, mode, n, dtype, ball):
    print(f"[case] tiles {case} {mode} {n} {dtype}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, sphere=ball, tau=0.1)
    want = state(n, 7, addr_mode=2, **kw)
    for shape in SHAPES:
        same(state(n, 7, shape, **kw), want, f"launch {shape}")


# The AA odd step's row kernel runs on lattices above 512 MiB: rows of two,
# three and eight wavefronts, rows left over in the last workgroup of a plane
ROWS = [("tgv", "faithful", (512, 131, 40), "f64"), ("tgv", "faithful", (192, 201, 131), "f32"),
        ("tgv", "faithful", (128, 515, 160), "f16"), ("cavity", "config", (192, 101, 140), "f64"),
        ("cavity", "config", (128, 203, 201), "f32"), ("cavity", "config", (512, 67, 79), "f64")]


@pytest.mark.parametrize("case,mode,n,dtype", ROWS)
def test_row_kernel_equals_arrays(case, mode, n, dtype):
    print(f"[case] rows {case} {n} {dtype}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, storage="aa")
    want = state(n, 5, addr_mode=2, **kw)
    for shape in (None, (512, 1, 0, 0)):
        same(state(n, 5, shape, **kw), want, f"launch {shape}")


@pytest.mark.parametrize("dtype,storage", [("f64", "pull"), ("f64", "aa"), ("f32", "pull"), ("f16", "aa")])
def test_ensemble_mixes_layouts(dtype, storage):
    """Members in plane tiles and in arrays (planes below 512 cells), periodic
    and cavity, ragged: each steps as the single domain does."""
    from imexlb_amd import LBM, Ensemble
    print(f"[case] ensemble layouts {dtype} {storage}", flush=True)
    sizes = [(0, 20, 21, 7), (1, 45, 37, 5), (0, 33, 31, 6), (1, 12, 10, 9), (0, 64, 64, 3), (1, 129, 9, 4)]
    doms = [dict(case_id=c, nx=x, ny=y, nz=z, tau0=0.05 + 0.01 * k, rho0=1.0, u0=0.05, lid_u=0.08)
            for k, (c, x, y, z) in enumerate(sizes)]
    want = []
    for d in doms:
        g = LBM(d["nx"], d["ny"], d["nz"], d["tau0"], u0=0.05, lid_u=0.08, case="cavity" if d["case_id"] else "tgv",
                mode="config" if d["case_id"] else "faithful", dtype=dtype, storage=storage, addr_mode=2)
        g.Initialize()
        g.step(7)
        want.append(g.moments())
        g.close()
    e = Ensemble(doms, dtype=dtype, storage=storage)
    for launch in (None, (64, 1, 24), (192, 2, 0), (512, 1, 8)):
        if launch:
            e.set_launch(*launch)
        for mode in ("persistent", "graph", "per_domain"):
            e.Initialize()
            e.step(7, mode=mode)
            for k in range(len(doms)):
                for name, a, b in zip("puvw", want[k], e.moments(k)):
                    assert np.array_equal(a, b), f"member {k} {name}, launch {launch}, {mode}"
    e.close()


# (8, 8): the smallest tiled plane; (7, 9): the largest that is not; (13, 5),
# (2, 33): one cell more than a wavefront; (9, 13), (16, 31): ragged
SMALL_PLANES = [(8, 8, 3), (7, 9, 4), (13, 5, 6), (2, 33, 5), (9, 13, 2), (16, 31, 3)]


@pytest.mark.parametrize("n", SMALL_PLANES)
@pytest.mark.parametrize("case,mode,dtype,storage", [("tgv", "faithful", "f64", "pull"), ("tgv", "faithful", "f32", "aa"),
                                                     ("cavity", "config", "f64", "aa"), ("cavity", "config", "f16", "pull"),
                                                     ("cavity", "faithful", "f64", "pull")])
def test_small_planes_equal_arrays(n, case, mode, dtype, storage):
    print(f"[case] small planes {case} {mode} {n} {dtype} {storage}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, storage=storage, tau=0.1)
    for steps in (6, 7):
        want = state(n, steps, addr_mode=2, **kw)
        for shape in (None, (128, 2, 1, 0), (64, 1, 0, 1)):
            same(state(n, steps, shape, **kw), want, f"{steps} steps, launch {shape}")


# both accesses of plane tiles (nt_loads), on both sides of the rule that chooses
@pytest.mark.parametrize("n,dtype,storage", [((40, 41, 39), "f64", "pull"), ((24, 40, 21), "f64", "aa"),
                                             ((33, 31, 30), "f32", "pull"), ((64, 64, 9), "f16", "aa")])
@pytest.mark.parametrize("case,mode", [("tgv", "faithful"), ("cavity", "config")])
def test_plain_and_non_temporal_agree(n, dtype, storage, case, mode):
    print(f"[case] accesses {case} {n} {dtype} {storage}", flush=True)
    kw = dict(case=case, mode=mode, dtype=dtype, storage=storage)
    want = state(n, 7, addr_mode=2, **kw)
    for nt in (0, 1):
        same(state(n, 7, (64, 1, 1, nt), **kw), want, f"nt {nt}")
    same(state(n, 7, **kw), want, "default")


# beyond the last-level cache a placement search times plane tiles and arrays
@pytest.mark.parametrize("n,dtype,storage", [((96, 96, 90), "f64", "pull"), ((160, 128, 131), "f32", "aa")])
def test_placement_searches_over_both_layouts_keep_results(n, dtype, storage):
    from imexlb_amd import LBM
    print(f"[case] searches {n} {dtype} {storage}", flush=True)
    want = state(n, 7, dtype=dtype, storage=storage)
    g = LBM(*n, 0.06, u0=0.05, dtype=dtype, storage=storage)
    for search in (lambda: g.tune_placement_window(slack_gib=8 / 1024, step_gib=4 / 1024, steps=4),
                   lambda: g.tune_placement(3, steps=4),
                   lambda: g.tune_placement_window(slack_gib=4 / 1024, step_gib=4 / 1024, steps=4)):
        kept, ms = search()
        assert all(m > 0 for m in ms) and ms[kept] == min(ms)
        g.Initialize()
        g.step(7, 3)
        same((g.get_f(), g.moments()), want, "after a search")
    g.step(32, 32)  # a graph recorded on the kept layout
    h = LBM(*n, 0.06, u0=0.05, dtype=dtype, storage=storage)
    h.Initialize()
    h.step(39, 39)
    for a, b in zip(g.moments(), h.moments()):
        assert np.array_equal(a, b)
    g.close()
    h.close()
