"""bench.py's line for the expansions: per level, by the bytes that were counted."""
from types import SimpleNamespace

import bench


def test_expansions_per_level():
    args = SimpleNamespace(scale=24, edge_factor=16, seed=24)
    moved = bench.load_traffic("bfs_expand_traffic.json")["bytes_per_level"]
    r = bench.bfs_roofline(args, entries=10**9, vertices=10**7, ns=10**6, levels=10)
    # a launch is not a level: nothing is given per launch
    assert r["levels"] == 10 and r["avg_level_us"] == 100.0 and not any("launch" in k for k in r)
    # bytes moved, and not those that a pull round skips
    assert r["traffic"] == moved and abs(r["achieved"] - moved / 1e-4 / 1e9) < 0.1
    assert r["topdown_bytes_per_level"] == 428 * 10**6
    assert "bfs_small_kernel" in r["kernel"]


def test_no_counters_for_another_workload():
    r = bench.bfs_roofline(SimpleNamespace(scale=20, edge_factor=16, seed=24), 10**6, 10**5, 10**6, 10)
    assert r["achieved"] is None and r["frac"] is None and "l2_requests" not in r
