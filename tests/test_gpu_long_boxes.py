"""Boxes of few cells a plane and more planes than whole workgroups fit into one
launch (2^24 of 256 threads): Initialize writes every cell."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PI_R = 3.1415926


@pytest.mark.parametrize("n", [(2, 2, (1 << 24) + 5), (8, 8, (1 << 18) + 3), (5, 13, 20011), (12, 12, 3000), (16, 15, 4099)])
@pytest.mark.parametrize("dtype,storage", [("f16", "aa"), ("f64", "pull")])
def test_initialize_writes_every_cell(n, dtype, storage):
    from imexlb_amd import LBM
    print(f"[case] long box {n} {dtype} {storage}", flush=True)
    nx, ny, nz = n
    if nz > 1 << 23 and dtype == "f64":
        dtype, storage = "f32", "aa"
    u0 = 0.05
    g = LBM(nx, ny, nz, 0.1, u0=u0, dtype=dtype, storage=storage)
    g.Initialize()
    p = g.moments()[0]
    a, b, c = (np.arange(k) / k * 2.0 * PI_R for k in n)
    want = 1 / 3 + u0 * u0 / 16 * (np.cos(2 * a)[None, None, :] + np.cos(2 * b)[None, :, None]) * (np.cos(2 * c)[:, None, None] + 2)
    # sums and products of a few values of size one; the cosine's argument is below 13
    assert np.abs(p - want).max() < 1e-14
    # the populations carry the same fields: one step keeps the mass, to the storage's
    # relative rounding of what it holds, u0^2 against 1
    before = 3.0 * float(p.sum())
    g.step(2)
    _, mass = g.diagnostics()
    assert abs(mass / before - 1.0) < u0 * u0 * {"f64": 1e-12, "f32": 1e-6, "f16": 1e-2}[dtype] + 1e-12
    g.close()
