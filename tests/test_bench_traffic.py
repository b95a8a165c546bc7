"""bench.py's roofline.traffic (CPU): the figure of the layout that the run kept."""
import importlib.util
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_belongs_to_the_layout():
    spec = importlib.util.spec_from_file_location("bench_mod", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
        held = json.load(f)
    keys = {am: bench.traffic_key(512, "aa", {"addr_mode": am}) for am in (-1, 2)}
    assert keys[-1] != keys[2] and set(keys.values()) <= set(held)
    for k in keys.values():
        t = held[k]
        assert bench.traffic_from_profiles(k) == (t["bytes_per_launch"], t["ratio"], t["source"])
        assert abs(t["bytes_per_launch"] / t["algorithmic_bytes_per_launch"] - t["ratio"]) < 1e-9
    assert bench.traffic_from_profiles(bench.traffic_key(96, "pull", {"addr_mode": -1})) is None
