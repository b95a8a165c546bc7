"""The lattices' layout on the host (layout_units.cpp): plane tiles of every plane
size hold each population of each cell once, leave at most a sixteenth unused or
what rounding up to 128-byte lines leaves, and large lattices less."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_layout_units(tmp_path):
    exe = str(tmp_path / "layout_units")
    r = subprocess.run([HIPCC, "-std=c++17", "-O1", "--cuda-host-only", "-x", "hip",
                        os.path.join(ROOT, "tests", "layout_units.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split() == ["ok"], r.stdout
