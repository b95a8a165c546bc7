"""Fields and populations read back into host memory (readback.h): every value
in its place, for reads of one piece, of exactly the small limit, of several
pieces with a short last one, of single fields, and into pinned memory."""
import ctypes

import numpy as np
import pytest

from oracle.oracle import TGV, Oracle

pytestmark = pytest.mark.gpu

# 4 fields of 8 bytes: 24 cells; 2 MiB exactly; one plane above; pieces of 1 MiB
# with a short last one; pieces of 4 MiB
SIZES = [(2, 3, 4), (16, 16, 256), (16, 16, 257), (130, 67, 33), (200, 190, 140)]


def make(n):
    from imexlb_amd import LBM
    g = LBM(*n, 0.05, u0=0.05)
    o = Oracle(TGV, *n, tau0=0.05, u0=0.05)
    g.Initialize()
    o.Initialize()
    return g, o


@pytest.mark.parametrize("n", SIZES)
def test_fields_and_populations(n):
    print(f"[case] read-back {n}", flush=True)
    g, o = make(n)
    want = o.moments()
    for _ in range(2):
        for a, b in zip(want, g.moments()):
            assert np.array_equal(a, b)
    assert np.array_equal(o.get_f(), g.get_f())
    g.close()


@pytest.mark.parametrize("n", SIZES[1:4])
def test_single_fields_and_pinned_memory(n):
    from imexlb_amd._lib import dptr, lib
    print(f"[case] read-back single, pinned {n}", flush=True)
    g, o = make(n)
    want = o.moments()
    out = [np.full(g.shape, np.nan) for _ in range(4)]
    none = ctypes.POINTER(ctypes.c_double)()
    assert lib().imexlb_get_moments(g.h, none, dptr(out[1]), none, dptr(out[3])) == 0
    assert np.isnan(out[0]).all() and np.isnan(out[2]).all()
    assert np.array_equal(out[1], want[1]) and np.array_equal(out[3], want[3])
    # pinned memory of the runtime that the library is linked with
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    nbytes = out[0].nbytes
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * nbytes), 0) == 0
    pinned = np.frombuffer((ctypes.c_char * (4 * nbytes)).from_address(p.value), dtype=np.float64).reshape((4,) + g.shape)
    assert lib().imexlb_get_moments(g.h, *[dptr(a) for a in pinned]) == 0
    for a, b in zip(want, pinned):
        assert np.array_equal(a, b)
    g.close()
    del pinned
    assert hip.hipHostFree(p) == 0


# fields that end inside a 16-byte unit, and that start inside one in pinned
# memory's order: one kernel copies all four
@pytest.mark.parametrize("n", [(3, 3, 3), (5, 7, 3), (41, 39, 37)])
def test_fields_of_odd_cell_counts(n):
    print(f"[case] read-back odd {n}", flush=True)
    g, o = make(n)
    for a, b in zip(o.moments(), g.moments()):
        assert np.array_equal(a, b)
    assert np.array_equal(o.get_f(), g.get_f())
    g.close()
