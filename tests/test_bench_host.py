"""Host logic of bench.py, on the CPU: the one-GPU guard and the HBM-traffic arithmetic
that turns two rocprofv3 --pmc counter files into bytes per Heff application."""
import csv
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 2
    assert "one GPU only" in r.stderr
    assert r.stdout == ""


def write_counters(path, counter, rows):
    # rocprofv3 counter_collection.csv columns that the parser reads
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=["Dispatch_Id", "Kernel_Name", "Counter_Name", "Counter_Value"])
        w.writeheader()
        for d, (name, v) in enumerate(rows):
            w.writerow({"Dispatch_Id": d + 1, "Kernel_Name": name, "Counter_Name": counter, "Counter_Value": v})
            # another counter in the same file is ignored
            w.writerow({"Dispatch_Id": d + 1, "Kernel_Name": name, "Counter_Name": "GRBM_COUNT", "Counter_Value": 7})


@pytest.mark.parametrize("fetch_per_gib,write_per_gib", [(2.0, 1.0), (1.0, 1.0), (0.5, 1.25)])
def test_traffic_numbers(tmp_path, fetch_per_gib, write_per_gib):
    # a counter that reads fetch_per_gib GiB for the 1 GiB copy mark is scaled by its
    # inverse; only the dispatches between the two largest marks count, per application
    gib_kib = bench.COPY_MARK_DOUBLES * 8 / 1024.0
    steps = 3
    kread = [100.0, 250.0, 50.0] * steps       # KiB as the counter reads them
    kwrite = [40.0, 10.0, 5.0] * steps
    small_mark = ("elementwise_kernel small", 12.0)  # a torch copy before the marks: not a bracket
    fetch = [small_mark, ("copyBuffer", gib_kib * fetch_per_gib)] + [("k_tiles_fit", v) for v in kread] + \
            [("elementwise_kernel", gib_kib * fetch_per_gib), ("k_after", 1e9)]
    write = [small_mark, ("copyBuffer", gib_kib * write_per_gib)] + [("k_tiles_fit", v) for v in kwrite] + \
            [("elementwise_kernel", gib_kib * write_per_gib), ("k_after", 1e9)]
    fp, wp = str(tmp_path / "fetch.csv"), str(tmp_path / "write.csv")
    write_counters(fp, "FETCH_SIZE", fetch)
    write_counters(wp, "WRITE_SIZE", write)
    out = bench.traffic_numbers(fp, wp, steps)
    rd = sum(kread) / fetch_per_gib * 1024.0 / steps
    wr = sum(kwrite) / write_per_gib * 1024.0 / steps
    assert out["read_bytes"] == pytest.approx(rd, rel=1e-12)
    assert out["write_bytes"] == pytest.approx(wr, rel=1e-12)
    assert out["bytes_per_launch"] == pytest.approx(rd + wr, rel=1e-12)
    assert out["fetch_scale"] == pytest.approx(1.0 / fetch_per_gib, abs=1e-4)
    assert out["dispatches_per_application"] == 3
    assert out["applications"] == steps


def test_roofline_record_matrix_core_bound():
    # the middle-site product of the L=32 D=2000 benchmark as measured on one MI355X:
    # 16.7922 ms of kernels for F_H = 2.2925e11 flops over B_H = 7.2768e8 algorithmic bytes
    r = bench.roofline_record(229251582970.0, 727681104.0, 16.7922, 54519203899.42752, "profiles/x.json")
    assert r["bound"] == "mfma"           # 315 flop/B x 8 TB/s is far above 78.6 TFLOP/s
    assert r["peak"] == 78.6
    assert r["achieved"] == 13.6523
    assert r["frac"] == 0.1737
    assert r["traffic_over_B_H"] == 74.92
    assert r["unit"] == "TFLOP/s" and r["traffic_source"] == "profiles/x.json"


def test_roofline_record_hbm_bound():
    # 1 flop per byte: the bound is 8 TFLOP/s of HBM, and 1 TFLOP/s is 1/8 of it
    r = bench.roofline_record(1e9, 1e9, 1.0, None, None)
    assert r["bound"] == "hbm"
    assert r["peak"] == 8.0
    assert r["achieved"] == 1.0
    assert r["frac"] == 0.125
    assert r["traffic_over_B_H"] is None


def test_printed_record_is_short():
    # of a run's size: 60 sites in each of three forms
    sweep = {"seconds": 1234.567, "presolve_seconds": 1.234, "total_min_energy": -45.762898269479706,
             "heff_applications": 12345, "heff_applications_hi_only": 12345, "heff_flops": 1.5437882058412345e17,
             "heff_device_seconds": 1234.5678, "heff_tflops_sweep_average": 17.1234,
             "phase_seconds": {k: 123.456 for k in ("join", "prepare", "davidson", "split", "update", "total")},
             "sites": [{"site": q, "energy": -45.762898269479706, "products": 12, "heff_ms": 123.456,
                        "F_H": 154378820584.0} for q in range(60)],
             "delta_E_vs_fp64": 2.5437429940211587e-12, "speedup_vs_fp64": 0.926}
    sb = {"site": 15, "V": 186316, "F_H": 1.234e11, "B_H": 1.234e9, "ms_kernels": 10.1234, "ms_per_call": 10.1234,
          "tflops": 17.1234, "kernel_ms": [1.0, 2.0, 3.0], "plan_stats": {str(q): 10 ** 9 for q in range(16)}}
    out = {
        "metric": "Heff\u00b7x TFLOP/s + Davidson sweep time at L=32 D=2000; |\u0394E| vs FP64 \u22641e-8 Ha",
        "value": 17.1234, "unit": "TFLOP/s", "n_gpus": 1, "steps": 12345, "warmup": 5, "ms_per_step": 10.1234,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic",
        "config": {"workload": "w" * 160, "L": 32, "D": 2000, "davidson_rtol": 1e-5, "sweep_seconds_fp64": 1234.567},
        "roofline": bench.roofline_record(1.2345678901234e11, 1.2345678901234e9, 10.1234, 54512345678.9, "profiles/" + "t" * 40),
        "cpu_baseline": {"value": 0.123456789012345, "unit": "TFLOP/s", "cores": 256, "kind": "reference",
                         "sample": "s" * 500, "seconds_per_step": [1.0] * 30, "presolve_seconds": 1.0},
        "warm_up": {"seconds": 100.0}, "site_bench": sb,
        "sweep": {"fp64": sweep, "mixed": sweep, "mixed+learned": sweep},
        "n2_ccpvdz_published_point": {"seconds_per_sweep": 15.184, "energy": -109.28215523999137, "warm_up_seconds": 18.06,
                                      "heff_applications": 2108, "published": bench.N2_PUBLISHED, "speedup_vs_published": 14.4},
    }
    line = bench.json.dumps(bench.summary(out))
    assert len(line) < 2000
    got = bench.json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert got[k] == out[k]
    assert got["sweep"]["fp64"]["seconds"] == sweep["seconds"]
    # parts that a run left out
    short = dict(out, roofline=bench.roofline_record(1e11, 1e9, 10.0, None, None), cpu_baseline=None,
                 n2_ccpvdz_published_point=None, sweep={"fp64": sweep})
    assert "cpu_baseline" not in bench.summary(short) and bench.summary(short)["value"] == 17.1234
