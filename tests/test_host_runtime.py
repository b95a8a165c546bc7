"""The library's host code on a HIP runtime without a GPU (fake_hip.cpp): what it
allocates and launches, at sizes and limits that no test can afford on a device."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")

PREAMBLE = """
import ctypes, sys
F = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
F.fake_name.restype = ctypes.c_char_p
F.fake_grid.restype = F.fake_block.restype = F.fake_used.restype = F.fake_most_pinned.restype = ctypes.c_size_t
F.fake_room.argtypes = F.fake_paint.argtypes = [ctypes.c_size_t]
F.fake_cost.argtypes = [ctypes.c_char_p, ctypes.c_double]
import numpy as np
from imexlb_amd import LBM, Ensemble

def launches():
    out = [(F.fake_name(k).decode(), F.fake_grid(k), F.fake_block(k)) for k in range(F.fake_launches())]
    F.fake_forget()
    return out
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    r = subprocess.run([HIPCC, "-std=c++17", "--cuda-host-only", "-x", "hip", "-shared", "-fPIC",
                        os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(script, *args):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + textwrap.dedent(script), so, *map(str, args)],
                           cwd=ROOT, capture_output=True, text=True, timeout=110)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def test_initialize_of_long_thin_boxes(fake):
    """Boxes of few cells a plane and many planes: the launch stays within the 2^32
    work-items that HIP takes, and follows the cells, not the planes."""
    fake("""
    for n in [(2, 2, 1 << 24), (3, 5, 1 << 24), (9, 7, 1 << 24), (8, 8, 1 << 24), (5, 13, 1 << 24), (16, 16, 1 << 22)]:
        g = LBM(*n, 0.1, dtype="f16", storage="aa")
        launches()
        g.Initialize()
        (name, grid, block), = launches()
        assert "k_init" in name and grid * block < 2 * n[0] * n[1] * n[2] + 256, (n, grid, block)
        g.close()
    """)


@pytest.mark.parametrize("shape", [(512, 1, 1, 1), (512, 2, 0, 0), (256, 1, 1, 0)])
def test_wide_workgroups_on_small_planes(fake, shape):
    """A workgroup as wide as the caller asks stays within its plane: what idles
    doesn't count towards the 2^32 work-items that HIP takes."""
    fake("""
    shape = tuple(int(v) for v in sys.argv[2].split(","))
    for n in [(8, 8, 1 << 23), (8, 8, 1 << 24), (10, 10, 21000000), (128, 2, 8388000)]:
        g = LBM(*n, 0.1, dtype="f16", storage="aa")
        g.set_launch(*shape)
        g.Initialize()
        launches()
        g.step(2, 0)
        for name, grid, block in launches():
            assert grid * block < 2 * n[0] * n[1] * n[2] + 512, (n, name, grid, block)
        g.close()
    """, ",".join(map(str, shape)))


def test_autotune_on_small_planes(fake):
    fake("""
    g = LBM(8, 8, 1 << 23, 0.1, dtype="f16", storage="aa")
    g.autotune(steps=2)
    """)


def test_batched_launch_of_very_many_tiles(fake):
    """Members whose tiles at one workgroup each exceed a launch: the grid stays
    below it and walks them."""
    fake("""
    e = Ensemble([dict(case_id=0, nx=32, ny=17, nz=490000, tau0=0.1, rho0=1.0, u0=0.05, lid_u=0.0)] * 12,
                 dtype="f16", storage="aa")
    e.Initialize()
    launches()
    e.step(2, mode="persistent", moments_every=0)
    got = launches()
    assert len(got) == 2 and all(grid * block < 1 << 32 for _, grid, block in got), got
    """)


@pytest.mark.parametrize("n", [(24, 20, 16), (80, 64, 64)])
def test_reads_of_several_threads(fake, n):
    """Threads that read fields of one handle at once, small and in pieces, each get
    their own: a read only looks at the handle."""
    fake("""
    import threading
    from imexlb_amd._lib import dptr, lib
    n = tuple(int(v) for v in sys.argv[2].split(","))
    g = LBM(*n, 0.1)
    g.Initialize()
    F.fake_paint(32 << 20)
    F.fake_copy_delay(300)
    want = [float(a.flat[0]) for a in g.moments()]
    assert len(set(want)) == 4
    none = ctypes.POINTER(ctypes.c_double)()
    wrong = []

    def read(k, rounds):
        out = np.empty(g.shape)
        for _ in range(rounds):
            out[:] = -1
            rc = lib().imexlb_get_moments(g.h, *[dptr(out) if i == k else none for i in range(4)])
            if rc or (out != want[k]).any():
                wrong.append(k)

    def read_all():
        if any((a != v).any() for a, v in zip(g.moments(), want)):
            wrong.append("all")

    ts = [threading.Thread(target=read, args=(k, 6)) for k in range(4)] + [threading.Thread(target=read_all) for _ in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong
    """, ",".join(map(str, n)))


@pytest.mark.parametrize("n,mib", [((16, 16, 16), 1), ((45, 37, 51), 4), ((64, 64, 64), 8), ((128, 128, 96), 24)])
def test_a_read_pins_what_it_uses(fake, n, mib):
    """The first read of a handle pins no more than its pieces, and at most 24 MiB."""
    fake("""
    n = tuple(int(v) for v in sys.argv[2].split(","))
    g = LBM(*n, 0.1)
    g.Initialize()
    F.fake_paint(64 << 20)
    for _ in range(2):
        assert len({float(a.min()) for a in g.moments()} & {float(a.max()) for a in g.moments()}) == 4
    assert F.fake_most_pinned() <= int(sys.argv[3]) << 20, F.fake_most_pinned()
    """, ",".join(map(str, n)), mib)


@pytest.mark.parametrize("n", [(13, 5, 153846), (9, 8, 138889), (10, 13, 76923), (12, 12, 69444), (23, 23, 18904)])
@pytest.mark.parametrize("dtype,storage", [("f64", "pull"), ("f32", "aa"), ("f16", "pull")])
def test_memory_of_boxes_of_small_planes(fake, n, dtype, storage):
    """The default layout of a large box holds at most a twelfth more than arrays."""
    fake("""
    n = tuple(int(v) for v in sys.argv[2].split(","))
    used = []
    for am in (2, -1):
        g = LBM(*n, 0.1, dtype=sys.argv[3], storage=sys.argv[4], addr_mode=am)
        used.append(F.fake_used())
        assert g.info()["device_bytes"] <= used[-1]
        g.close()
        assert F.fake_used() == 0
    assert used[1] <= used[0] * 13 / 12, used
    """, ",".join(map(str, n)), dtype, storage)


# (case, mode, more): every allocation that follows the lattices
LATER = [("tgv", "faithful", "{}"), ("cavity", "faithful", "{}"), ("sphere", "faithful", "{}"),
         ("sphere", "config", "dict(sphere=(30.0, 20.0, 20.0, 5.0))")]


@pytest.mark.parametrize("case,mode,more", LATER)
def test_arrays_where_only_they_fit(fake, case, mode, more):
    """A box whose arrays fit in the memory there is, and whose tiles do not, runs in
    arrays, whichever allocation is the one that fails; a box that fits neither way is
    refused and leaves nothing behind."""
    fake("""
    from imexlb_amd import ImexlbError
    kw = dict(case=sys.argv[2], mode=sys.argv[3], **eval(sys.argv[4]))
    n = (97, 41, 50)  # 3977 cells a plane: tiles hold 4096
    used = {}
    for am in (2, -1):
        g = LBM(*n, 0.1, addr_mode=am, **kw)
        used[am] = F.fake_used(), g.info()["device_bytes"]
        g.close()
    assert used[-1][0] > used[2][0] * 1.02
    for room in np.linspace(used[2][0], used[-1][0], 40):
        F.fake_room(int(room))
        g = LBM(*n, 0.1, **kw)
        assert g.info()["device_bytes"] == used[-1 if int(room) == used[-1][0] else 2][1]
        g.Initialize()
        g.step(2)
        g.close()
        assert F.fake_used() == 0
    for room in np.linspace(0, used[2][0] - 1, 40):
        F.fake_room(int(room))
        try:
            LBM(*n, 0.1, **kw)
            assert False, room
        except ImexlbError as e:
            assert e.status == -3, e
        assert F.fake_used() == 0
    """, case, mode, more)


def test_ensemble_in_arrays_where_only_they_fit(fake):
    fake("""
    from imexlb_amd import ImexlbError
    doms = [dict(case_id=k % 2, nx=97, ny=41, nz=20 + k, tau0=0.1, rho0=1.0, u0=0.05, lid_u=0.1) for k in range(3)]
    cells = sum(d["nx"] * d["ny"] * d["nz"] for d in doms)
    arrays = cells * (2 * 27 + 4) * 8 + (1 << 20)
    e = Ensemble(doms, dtype="f64")
    tiles = F.fake_used()
    e.close()
    assert F.fake_used() == 0 and tiles > arrays, (F.fake_used(), tiles, arrays)
    for room in np.linspace(arrays, tiles, 30):
        F.fake_room(int(room))
        e = Ensemble(doms, dtype="f64")
        e.Initialize()
        e.step(2)
        e.close()
        assert F.fake_used() == 0
    F.fake_room(cells * 58 * 8)
    try:
        Ensemble(doms, dtype="f64")
        assert False
    except ImexlbError:
        pass
    assert F.fake_used() == 0
    """)


def test_tuned_shapes_are_kept_by_layout(fake, tmp_path):
    """A cached launch shape serves handles of the layout it was timed on: not the
    other layout, and no line that names none is taken."""
    fake("""
    cache = sys.argv[2]

    def tune(am, **kw):
        g = LBM(66, 40, 30, 0.1, addr_mode=am, **kw)
        launches()
        c = g.autotune(cache, steps=2)
        timed = any("k_fused" in name or "k_tiled" in name for name, _, _ in launches())
        g.close()
        return c, timed

    F.fake_cost(b"k_fused_pair", 1e-3)  # two adjacent cells: faster, in arrays only
    F.fake_cost(b"k_init", 0.0)
    for p in (b"k_fusedI", b"k_tiled"):
        F.fake_cost(p, 2e-3)
    arrays, timed = tune(2)
    assert timed and arrays[1] == 3, arrays
    tiles, timed = tune(-1)
    assert timed and tiles[1] != 3, tiles
    assert tune(2) == (arrays, False) and tune(-1) == (tiles, False)
    keys = [line.split('"')[3] for line in open(cache)]
    assert len(set(keys)) == 2
    # lines of before, which say nothing of the layout
    with open(cache, "w") as f:
        for k in keys:
            f.write('{"key": "%s", "block": 448, "cpt": 1, "third": 0, "ntl": 0, "ms": 0.1}' % k.rsplit("_", 1)[0] + chr(10))
    for am in (2, -1):
        c, timed = tune(am)
        assert timed and c[0] != 448, c
    """, tmp_path / "cache.jsonl")


def test_tuned_ensemble_shapes_are_kept_by_layout(fake, tmp_path):
    """Two ensembles of equal counts, one of members in tiles and one in arrays."""
    fake("""
    cache = sys.argv[2]
    for nx, ny, nz in ((32, 32, 16), (16, 16, 64)):
        e = Ensemble([dict(case_id=0, nx=nx, ny=ny, nz=nz, tau0=0.1, rho0=1.0, u0=0.05, lid_u=0.1)] * 2)
        e.Initialize()
        for again in (False, True):
            launches()
            e.autotune(cache, steps=2)
            assert any("k_ensemble" in name for name, _, _ in launches()) != again
        e.close()
    """, tmp_path / "cache.jsonl")


@pytest.mark.parametrize("n,kw,block", [
    ((512, 256, 256), dict(case="sphere", mode="config", sphere=(128.0, 128.0, 128.0, 20.0), dtype="f16"), 192),
    ((128, 128, 128), dict(case="cavity", mode="config", storage="aa"), 256),
    ((32, 32, 32), dict(), 64),
    ((40, 40, 40), dict(block=448), 448)])
def test_autotune_times_the_untuned_shape(fake, n, kw, block):
    """Whatever shape a handle has by default is among those that the tuner times."""
    fake("""
    n, kw, block = eval(sys.argv[2])
    g = LBM(*n, 0.1, **kw)
    g.Initialize()
    launches()
    g.step(2, 0)
    untuned = launches()[-1][2]
    assert untuned == block, untuned
    g.set_launch(320, 1, 1, 1)
    launches()
    g.autotune(steps=2)
    timed = {b for name, _, b in launches() if "k_fused" in name or "k_tiled" in name}
    assert {64, 128, 256, 512, block} <= timed, timed
    """, repr((n, kw, block)))


SEARCHES = {"trials": "g.tune_placement(3, steps=2)", "window": "g.tune_placement_window(4, 2, steps=2)"}


@pytest.mark.parametrize("search", SEARCHES)
def test_placement_searches_try_both_layouts_from_either(fake, search):
    """A search times tiles and arrays at each place whichever the handle has, keeps the
    faster one, and accounts for what it holds."""
    fake("""
    def faster(part):
        for p in (b"k_fusedI", b"k_tiled"):
            F.fake_cost(p, 1e-3 if p == part else 2e-3)

    def kept():
        launches()
        g.Initialize()
        g.step(2, 0)
        return {name.split("I")[0].split("k_")[1] for name, _, _ in launches() if "k_init" not in name}

    for storage in ("aa", "pull"):
        g = LBM(200, 200, 100, 0.1, storage=storage)
        assert kept() == {"tiled"}
        own = g.info()["block"], g.info()["nt_loads"]
        for part in (b"k_fusedI", b"k_tiled", b"k_fusedI", b"k_fusedI", b"k_tiled"):
            faster(part)
            SEARCH
            assert kept() == {part.decode()[2:].split("I")[0]}, (storage, part)
            i = g.info()
            assert (i["block"], i["nt_loads"]) == (own if part == b"k_tiled" else (256, 1)), i
            assert 0 <= F.fake_used() - i["device_bytes"] < 1 << 20
        # the caller's own shape stays
        g.set_launch(320, 1, 1, 0)
        faster(b"k_fusedI")
        SEARCH
        assert g.info()["block"] == 320 and g.info()["nt_loads"] == 0
        g.close()
        assert F.fake_used() == 0
    """.replace("SEARCH", SEARCHES[search]))


@pytest.mark.parametrize("search", SEARCHES)
def test_placement_searches_of_lattices_in_the_last_level_cache(fake, search):
    """Their place in HBM hardly counts: the search times the handle's layout only."""
    fake("""
    for n in ((32, 32, 32), (40, 40, 40), (64, 64, 64)):
        g = LBM(*n, 0.1)
        launches()
        SEARCH
        assert not any("k_fused" in name for name, _, _ in launches()), n
        g.close()
    """.replace("SEARCH", SEARCHES[search]))


@pytest.mark.parametrize("search", SEARCHES)
def test_placement_searches_with_room_for_arrays_only(fake, search):
    """Where a further lattice fits in arrays and not in tiles, arrays are searched, as
    they were before there were tiles."""
    fake("""
    F.fake_cost(b"k_fusedI", 1e-3)
    F.fake_cost(b"k_tiled", 2e-3)
    n = (97, 41, 3000)
    g = LBM(*n, 0.1, storage="aa", addr_mode=2)
    arrays = g.info()["device_bytes"]
    g.close()
    g = LBM(*n, 0.1, storage="aa")
    tiles = g.info()["device_bytes"]
    assert tiles > arrays * 1.02
    lattice = arrays - n[0] * n[1] * n[2] * 32
    F.fake_room(F.fake_used() + lattice + (2 << 30) + (1 << 20) + SLACK)
    SEARCH
    assert g.info()["device_bytes"] < tiles + (2 << 30)
    launches()
    g.Initialize()
    g.step(2, 0)
    assert any("k_fused" in name for name, _, _ in launches())
    """.replace("SEARCH", SEARCHES[search]).replace("SLACK", "(4 << 30) + (1 << 20)" if search == "window" else "0"))


def test_info_names_the_layout(fake):
    """imexlb_get_info: no address mode in plane tiles, where cells per thread 3 is 1."""
    fake("""
    for am, shape, want in ((-1, 1, (-1, 1)), (-1, 2, (-1, 2)), (-1, 3, (-1, 1)), (2, 3, (2, 3)), (1, 3, (1, 1))):
        for how in ("config", "set_launch"):
            g = LBM(48, 40, 32, 0.1, addr_mode=am, cells_per_thread=shape if how == "config" else 0)
            if how == "set_launch":
                g.set_launch(128, shape, 1, 1)
            i = g.info()
            assert (i["addr_mode"], i["cells_per_thread"]) == want, (am, shape, how, i)
            g.close()
    assert LBM(48, 40, 32, 0.1, stride_pad=256).info()["addr_mode"] == 2
    """)
