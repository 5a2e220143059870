"""bench.py's HBM traffic of the cell kernels: summed over whichever tier-0 kernel
a launch took, and reported only from a record of the kernels that run now."""
import csv
import json

import pytest

import bench


def counters(path, counter, dispatches):
    path.mkdir()
    with open(path / "run_counter_collection.csv", "w", newline="") as f:
        w = csv.DictWriter(f, ["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        w.writeheader()
        for i, (name, kib) in enumerate(dispatches):
            w.writerow({"Dispatch_Id": i, "Kernel_Name": name, "Counter_Name": counter, "Counter_Value": kib})
    return str(path)


@pytest.mark.parametrize("tier0", ["cell_group_kernel", "cell_group_small_kernel"])
def test_traffic_per_launch(tmp_path, monkeypatch, tier0):
    monkeypatch.setattr(bench, "TRAFFIC_PATH", str(tmp_path / "traffic.json"))
    step = [(f"pg::{tier0}(pg::CellParams)", 1000.0), ("pg::cell_group_mid_kernel(pg::CellParams)", 24.0),
            ("pg::knn_kernel<16>(long)", 5000.0)]
    copy = [(bench.COPY_KERNEL, 2048.0)]
    fetch = counters(tmp_path / "fetch", "FETCH_SIZE", 2 * step + [(bench.COPY_KERNEL, 1024.0)])
    write = counters(tmp_path / "write", "WRITE_SIZE", 2 * step + copy)
    rec = bench.summarize_pmc(fetch, write, 2, "w", "cmd")
    assert rec["bytes_per_launch"] == 2 * 1024 * 1024 + 1024 * 1024  # (the copy reads as half its bytes in FETCH_SIZE)
    assert bench._traffic_record("w")["bytes_per_launch"] == rec["bytes_per_launch"]


def test_a_record_of_other_kernels_is_not_reported(tmp_path, monkeypatch):
    path = tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "TRAFFIC_PATH", str(path))
    path.write_text(json.dumps({"w": {"bytes_per_launch": 5, "kernels": ["cell_group_kernel", "cell_group_exact_kernel"]}}))
    assert bench._traffic_record("w") is None and bench._traffic_record("other") is None
    path.write_text(json.dumps({"w": {"bytes_per_launch": 5, "kernels": list(bench.CELL_KERNELS)}}))
    assert bench._traffic_record("w")["bytes_per_launch"] == 5
