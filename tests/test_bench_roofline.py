"""The bench line's roofline: a fraction of the peak that bounds the launch, never above one."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_roofline_is_a_fraction():
    sys.path.insert(0, ROOT)
    import bench

    launches = json.load(open(os.path.join(ROOT, "profiles", "traffic_intersect_incoherent_1024.json")))["launches"]
    for p in launches:
        ms = p["kernel_trace_avg_ms"]
        r = bench.roofline(ms, p["algorithmic_bytes_per_launch"], p["hbm_bytes_per_launch"],
                           bench.valu_from_profiles(p["launch"]))
        assert r["bound"] == "valu_issue" and 0 < r["frac"] < 1
        assert abs(r["achieved"] * ms * 1e6 / p["sq_insts_valu_per_launch"] - 1) < 1e-3
        assert 0 < r["hbm"]["frac"] < 1 and r["algorithmic_gbs"] > r["hbm"]["achieved"]
        # without counters: the algorithmic bytes, a fraction only where HBM could bring them
        r = bench.roofline(ms, p["algorithmic_bytes_per_launch"], None, None)
        assert r["bound"] == "hbm" and r["frac"] is None and r["hbm"] is None
    assert bench.valu_from_profiles("variant=3") is None
    assert bench.roofline(10.0, 8e9, None, None)["frac"] == 0.1
