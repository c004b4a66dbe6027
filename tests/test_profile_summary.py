"""The HBM traffic that bench.py reports for a kernel is the one of the shape the workload launched most, the form of the
substep kernel with several levels per thread among its shapes."""
import csv
import os

from cppwrf_amd import profile_summary as PS
from cppwrf_amd.serving import alloc_elems


def _counters(d, counter, rows):
    d.mkdir()
    with open(d / "1_counter_collection.csv", "w", newline="") as f:
        w = csv.DictWriter(f, ["Kernel_Name", "Counter_Name", "Counter_Value"])
        w.writeheader()
        for name, value, n in rows:
            for _ in range(n):
                w.writerow({"Kernel_Name": f"void mi_fp32::(anonymous namespace)::{name}(mi_fp32::Args, double, int, int)",
                            "Counter_Name": counter, "Counter_Value": value})


def test_traffic_of_the_launched_substep_form(tmp_path, monkeypatch):
    monkeypatch.setattr(os, "environ", dict(os.environ))  # bench sets OpenMP's thread binding for its own process
    import bench
    n3 = alloc_elems(20, 16, 12)
    copy = (5 * 4 * n3 + 8 * (n3 // 13)) / 1024.0  # KiB, so both scale factors are 1
    rows = [("k_copy_step", copy, 3), ("k_acoustic<8, 64>", 1000.0, 4), ("k_acoustic_levels<8, 2, true>", 700.0, 30),
            ("k_uv<false>", 50.0, 30)]
    for c in ("FETCH_SIZE", "WRITE_SIZE"):
        _counters(tmp_path / c, c, rows)
    (tmp_path / "profiles").mkdir()
    (tmp_path / "profiles" / "t.md").write_text(PS.traffic(str(tmp_path / "FETCH_SIZE"), str(tmp_path / "WRITE_SIZE"), "20x16x12"))
    monkeypatch.setattr(bench, "HERE", str(tmp_path))
    got = bench.measured_traffic("t.md", "acoustic", "fp32")
    assert got["shape"] == "levels:8x2xtrue" and got["bytes"] == 2 * 700 * 1024
    assert bench.measured_traffic("t.md", "uv", "fp32")["bytes"] == 2 * 50 * 1024
