"""bench.py from the command line: the refusals that need no GPU, and on the GPU the switches that change which kernels
a step launches (each must still produce one JSON line with the contract's fields)."""
import argparse
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _bench(*flags, timeout=280):
    return subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), *flags], capture_output=True, text=True,
                          timeout=timeout, cwd=ROOT)


def test_more_than_one_gpu_is_refused_with_a_message():
    r = _bench("--gpus", "2")
    assert r.returncode == 2
    assert "one GPU" in r.stderr and r.stdout.strip() == ""


def test_counter_figures_of_other_kernels_are_not_used(tmp_path, monkeypatch):
    monkeypatch.syspath_prepend(ROOT)
    import bench

    args = argparse.Namespace(weight_stream=False, transposed_copies=False, grad_transposed_copy=False, fp8_activations=False)
    summary = tmp_path / "counters.txt"
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(summary))
    for kernels, flags, used in ((bench.kernel_digest(), "default", True), ("0" * 16, "default", False), (None, "default", False),
                                 (bench.kernel_digest(), "weight_stream", False)):
        summary.write_text("[bench-readable]\nflags = %s\n%sgemm_fetch_bytes_per_step = 4e9\ngemm_write_bytes_per_step = 1e9\n"
                           "quant_fetch_bytes_per_launch = 3e7\nquant_write_bytes_per_launch = 2e7\n" % (flags, f"kernels = {kernels}\n" if kernels else ""))
        got = bench.read_traffic(args)
        assert (got["gemm"], got["quant"]) == ((5e9, 5e7) if used else (None, None))
        assert ("note" in got["source"]) != used


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [("--fp8-activations",), ("--transposed-copies", "--grad-transposed-copy"), ("--no-graph",)])
def test_step_variants_print_one_contract_line(flags):
    r = _bench(*flags, "--steps", "2", "--warmup", "1", "--no-cpu-baseline")
    assert r.returncode == 0, r.stderr[-2000:]
    lines = [l for l in r.stdout.splitlines() if l.startswith("{")]
    assert len(lines) == 1
    d = json.loads(lines[0])
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config", "roofline"):
        assert key in d, key
    assert d["n_gpus"] == 1 and d["steps"] == 2 and d["value"] > 0 and d["vs_baseline"] is None
    assert d["roofline"]["bound"] == "mfma" and 0 < d["roofline"]["frac"] < 1
    assert d["config"]["launch"] == ("eager" if "--no-graph" in flags else "hip graph replay"), d["config"]["launch_note"]
    if "--fp8-activations" not in flags:
        assert d["verified"] and max(d["verified"]["worst_rel_l2"].values()) <= 1e-3
