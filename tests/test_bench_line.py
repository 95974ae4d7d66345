"""The benchmark's one line: valid JSON with the headline's figures exact, short enough to be kept whole (a line of the
workload's real structure in full has about 11,000 characters, of which readers kept the end)."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def _accuracy():
    q = {"max": 1.2345678901234e-06, "p999": 1.2345678901234e-07}
    return {"S11_rel": q, "floored_elem": q, "norm_elem": q, "floored_per_element_max": [1.2345678901234e-06] * 16,
            "failing_bins": 125847, "bins": 162360, "meets_gate": False,
            "first_failing": [{"theta_deg": 38.5000010713601, "phi_deg": 228.000006344678}] * 8}


def _plan():
    roof = {"bound": "valu", "achieved": 52.466812345678, "peak": 157.3, "unit": "TFLOP/s", "frac": 0.33354612345678,
            "traffic": 29844864666.4147, "kernel": "k_sweep<1,32,1> (estimate) + k_sweep<4,16,1> (listed bins)",
            "kernel_ms": 385.00912345678, "flop_per_beam_bin": 250.0, "beam_bins_per_launch": 694694689920}
    return {"value": 209766019429.74475, "unit": "beam·bin/s", "ms_per_step": 385.1945480000012, "steps": 2,
            "speedup_vs_fp64_plain": 2.5929571178665487, "autotune_ms": {f"{t}x{b}": 12.345678901 for t in (8, 16, 32)
                                                                         for b in (1, 2)},
            "tiles": {"beams_per_tile": 32, "bins_per_thread": 1, "chunks": 2, "workgroups": 1280}, "roofline": roof,
            "accuracy": _accuracy()}


def test_line_is_whole():
    text = "w" * 300
    base = {"value": 71929999.123456789, "unit": "beam·bin/s", "cores": 16, "kind": "port", "sample": text}
    out = {"metric": bench.METRIC, "unit": "beam·bin/s", "n_gpus": 1, "steps": 20, "warmup": 5, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "data": "synthetic", "dtype": "f64", **_plan(),
           "config": {"workload": text, "beams": 4296849, "beams_per_orientation": [4954, 5763], "precision": "fp64_fast",
                      "step": text[:80], "records": text[:80]}, "cpu_baseline": base}
    gate3 = {k: _accuracy() for k in ("fp64", "fp64_fast", "mixed")}
    sections = {"mixed": _plan(), "mixed_gated": {**_plan(), "refined_bins": 100114},
                "stress": {"workload": text, "beams": 200000, **{k: _plan() for k in ("mixed", "fp64_fast", "fp64")},
                           "vs_fp64_model": {"model": text[:60], **gate3}, "cpu_baseline": base},
                "large_column": {"workload": text, "fp64_plain": {"value": 8.1e10 / 7, "ms": 998.8123456789},
                                 "fp64_fast": _plan(), "mixed": _plan(), "vs_fp64_model": {"model": text[:60], **gate3}},
                "adjoint": {"workload": text, **{p: {k: 152.6361234567 for k in (
                    "forward_ms", "backward_ms", "backward_over_forward", "forward_kernel_ms", "adjoint_kernel_ms")}
                    for p in ("mixed", "fp64")}},
                "dropin": {"workload": text, **{p: {"diff_main_ms": 4.16353123456, "diffraction_ms_per_beam": 0.224954123}
                                                for p in ("fp64", "fp64_fast", "mixed")}},
                "visibility": {**_plan(), "config": {"workload": text}, "cpu_baseline": {**base, "gpu_over_cpu": 168.7}}}
    line = bench.json_line(out, sections)
    assert "\n" not in line and len(line) <= 6000, len(line)
    assert len(json.dumps({**out, **sections})) > 10000
    d = json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config", "cpu_baseline"):
        assert d[k] == out[k] or k == "cpu_baseline", k
    assert d["roofline"]["kernel_ms"] == 385.009 and d["accuracy"]["meets_gate"] is False
    assert d["stress"]["fp64_fast"]["ms_per_step"] == 385.195 and d["mixed_gated"]["refined_bins"] == 100114
    assert d["large_column"]["vs_fp64_model"]["fp64_fast"]["floored_elem"]["max"] == 1.23457e-06
