"""bench.py --traffic-update on counter files made here (no GPU): the traffic of
a query is that of all the kernels that answer it, and the key names the
kernel."""
import argparse
import csv
import json
import types

import pytest

import bench


def counters(path, rows):
    path.mkdir()
    with open(path / "x_counter_collection.csv", "w", newline="") as f:
        out = csv.DictWriter(f, ["Counter_Name", "Kernel_Name", "Dispatch_Id", "Counter_Value"])
        out.writeheader()
        for i, (counter, kernel, value) in enumerate(rows):
            for half in (1, 3):   # a dispatch's counter comes in parts
                out.writerow(dict(Counter_Name=counter, Kernel_Name=f"void mlmq::{kernel}<false>(Args)",
                                  Dispatch_Id=i, Counter_Value=value * half / 4))


@pytest.mark.parametrize("waves,kernel,launches", [
    (1, "sssp_persistent_kernel", [("sssp_persistent_kernel", 400)]),
    (10, "region_solver_kernel", [("region_solver_kernel", 400)]),
    (8, "push_kernel", [("push_kernel", 20)] * 15 + [("pull_kernel", 60)] + [("push_kernel", 20)] * 2)])
def test_bytes_of_a_query(tmp_path, capsys, waves, kernel, launches):
    assert bench.SOLVERS[bench.solver_of(dict(waves=waves * 64, work_blocks=64))][0] == kernel
    args = types.SimpleNamespace(buckets=2, window=2, l2_batch=8, min_read=8, l1_pop=32, l1_donate=0,
                                 light_split=0, stale_check=2, prefetch=1)
    key = bench.traffic_key("w", "L1SLF_L2DQ", 100, args, 64, kernel)
    assert kernel in key
    line = dict(roofline=dict(traffic_key=key, kernel=kernel), device_ms=dict(mean=1.5))
    (tmp_path / "line").write_text("log\n" + json.dumps(line) + "\n")
    for name, counter in (("f", "FETCH_SIZE"), ("w", "WRITE_SIZE")):
        queries = [(counter, "reset_kernel", 1000), *((counter, k, v) for k, v in launches)] * 3
        counters(tmp_path / name, queries)
        counters(tmp_path / ("c" + name), [(counter, "copy_u32_kernel", 512)] * 2)
    out = tmp_path / "traffic.json"
    bench.traffic_update(argparse.Namespace(
        traffic_update=[str(tmp_path / x) for x in ("line", "f", "w", "cf", "cw")],
        copy_bytes=512 * 1024, traffic_json=str(out)))
    entry = json.loads(out.read_text())[key]
    assert entry["bytes_per_launch"] == 2 * 400 * 1024 and entry["dispatches"] == [3, 3]
    assert bench.load_traffic(str(out), key) == entry["bytes_per_launch"]
    capsys.readouterr()
