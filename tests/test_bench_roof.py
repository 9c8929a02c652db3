"""bench.py's roofline entry of the cross-term kernel: priced by its arithmetic alone.
Bytes behind the L2 are mostly the Infinity Cache's and rise when the L2 is used
worse, so more of them must not read as nearness to a roof."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_traffic_is_no_roof():
    few = bench.cross_roofline(2.0e11, 4.0e10, 9.3, 45.0e9, False)
    many = bench.cross_roofline(2.0e11, 4.0e10, 9.3, 66.0e9, False)
    none = bench.cross_roofline(2.0e11, 4.0e10, 9.3, None, True)
    for r in (few, many, none):
        assert r["bound"] == "valu" and r["unit"] == "TFLOP/s"
        assert abs(r["achieved"] - 2.0e11 / 9.3e-3 / 1e12) < 1e-9
        assert abs(r["frac"] - r["achieved"] / 78.6) < 1e-12
    assert abs(many["traffic_gbs"] / few["traffic_gbs"] - 66 / 45) < 1e-9
    assert "traffic_gbs" not in none and none["arith"] == "f32"
