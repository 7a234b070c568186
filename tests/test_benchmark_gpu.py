"""The operator benchmark on the GPU: one cell of the launch-shape sweep and one line of the
table mode run end to end (tiny problems; this checks the tool, not the numbers)."""
import csv

import pytest

pytestmark = pytest.mark.gpu


def test_one_sweep_cell_and_one_table_line(tmp_path, capsys):
    from msd_pytorch_amd import _native, benchmark_ops as bo
    out = tmp_path / "sweep.csv"
    rc = bo.main(["--sweep", "--ndim", "3", "--size", "16", "16", "64", "--channels", "5", "--dilations", "2",
                  "--ops", "forward", "backward_xkb", "--limit", "3", "--trials", "1", "--csv", str(out)])
    assert rc == 0
    rows = list(csv.DictReader(open(out)))
    assert len(rows) == 2 * 4 and rows[0]["setting"] == "default" and rows[4]["setting"] == "default"
    assert {r["op"] for r in rows} == {"forward", "backward_xkb"}
    assert all(float(r["us"]) > 0 and float(r["GBps"]) > 0 for r in rows)
    text = capsys.readouterr().out
    assert "best" in text and "[4 settings]" in text
    # the sweep leaves every knob at the library default
    lib = _native.load()
    for key in bo.SWEEP_GRID["forward"][3]:
        assert lib.msd_set_tuning(key.encode(), -1) == 0
    rc = bo.main(["--ndim", "2", "--size", "128", "--channels", "3", "--dilations", "1", "--trials", "1"])
    assert rc == 0
    assert "forward" in capsys.readouterr().out


def test_the_traffic_of_other_launches_is_not_quoted(monkeypatch):
    """bench.py on its smallest workload: the step's kernels are the ones that its launches are compared by, and a summary taken with
    another number of them gives no figure."""
    import argparse

    import torch

    import bench
    from msd_pytorch_amd import _native
    args = argparse.Namespace(steps=2, warmup=1, graph=False, no_kernel_timing=False, tune=[], no_cpu_baseline=True)
    lib = _native.load()
    model = bench.make_model("A", torch)
    x, target = bench.make_data("A", torch)
    model.set_input(x)
    model.set_target(target)
    model.step_async(update=False)
    names = bench.step_kernels(model, torch)
    families = bench.FAMILIES["backward_xkb"]
    now = {f: sum(f in n for n in names) for f in families}
    assert now["pull_rows"] == now["sum_group"] == 1 and now["finish_back"] + now["spread_back"] == 9
    assert torch.isfinite(model.step_async(update=False) or model.loss)          # (eager steps go on)
    for extra, quoted in ((0, True), (1, False)):
        profiled = {**now, "pull_rows": now["pull_rows"] + extra}
        monkeypatch.setattr(bench, "profiled_traffic", lambda *a: ({c: (1e6, profiled if c == "backward_xkb" else {})
                                                                    for c in bench.FAMILIES}, "a summary"))
        roof = bench.measure("A", args, lib, torch, cpu=False)["roofline"]
        assert roof["kernel"] == "backward_xkb"
        assert (roof["traffic"] is not None) == quoted and ("traffic_note" in roof) != quoted
