"""The VALU bound that the benchmark's line reports is one that the kernel
cannot pass: by the rows in range of the shortened divisions (no GPU)."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_reported_bound_is_the_rows_in_range():
    # 8192^2 Van Leer has run at 27.1 Gcell-updates/s, above the bound of the general rows
    v = bench.valu_line(bench.valu_bound("MUSCLHancock", "VanLeer", "fp64", 27.1e9))
    assert v["achieved"] > v["general_rows"]["bound"]
    assert v["achieved"] < v["bound"] and v["frac"] < 1
    # 939 instructions at 4 cycles and 36 at 16 on 1 024 SIMDs at 2.4 GHz, 60 cells
    assert abs(v["bound"] - 1024 * 2.4e3 * 60 / (939 * 4 + 36 * 16)) < 0.1
    assert abs(v["frac"] - 27.1e3 / v["bound"]) < 1e-4
