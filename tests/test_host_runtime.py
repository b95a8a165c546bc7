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
F.fake_room.argtypes = [ctypes.c_size_t]
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
