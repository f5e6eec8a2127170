"""bench.py's one JSON line: whole in a reader's last LINE_LIMIT characters
with every leg of a default run in it, the top-level numbers untouched."""

from __future__ import annotations

import json

import bench


def _timing(ms, eager=False, covered=True):
    t = bench.Timer._summary([ms, ms * 1.01, ms * 0.987654321] * 2, [0.123456789012345], 1, covered, 1,
                             launches_per_trial=20, timing="hip graph replay")
    return {**t, "eager": _timing(ms * 1.1)} if eager else t


def _leg(ms, key="us_per_token", **extra):
    return {key: ms * 1e3, "timing": _timing(ms), "algorithmic_bytes": 105416192, "hbm_gbps": 3129.6045363439803,
            "hbm_frac": 0.39120056704299755, **extra}


def _line():
    stages = {"route": 0.005403750008554198, "phase1": 0.0223482656001579, "phase2": 0.012421515624737367}
    mode = {"k1": {**_leg(0.04058260023593903), "timing": _timing(0.04, eager=True), "stage_ms": stages},
            "k8": {**_leg(0.15972280502319336, distinct_pages=41.5, adjacent_overlap=0.09375, stage_ms=stages,
                          stage_note="n" * 200), "timing": _timing(0.16, eager=True)},
            "config0": _leg(0.0275, stage_ms=stages), "config1": _leg(0.02125, key="us_per_matvec")}
    cores = {"cores": 16, **{f"config{i}_{u}": 44259.7429999978 for i in range(3) for u in ("us_per_call", "runs")}}
    return {
        "metric": "MoE layer µs/token + achieved HBM GB/s (% peak) at K=1 and K=8, 1 MI355X",
        "value": 40.582600235939026, "unit": "us/token", "n_gpus": 1, "steps": 20, "warmup": 5,
        "ms_per_step": 0.04058260023593903, "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "d" * 90, "config": {"workload": "w" * 250, "timing": "t" * 300},
        "hbm_gbps": 2410.2325487113217, "hbm_frac": 0.30127906858891523, **mode, "other_mode": {"fast": mode},
        "variants": {f"k1_reference_layer_variant_{i}": _leg(0.0336, router="sqrt-softplus x 1.5", stage_ms=stages)
                     for i in range(9)},
        "prefill": _leg(0.72, key="ms_per_prefill", routing="r" * 80, official=_leg(0.74, key="ms_per_prefill")),
        "fp8_linear": {f"{n}_m{m}_{f}": _leg(0.0101, key="us", n=32768, k=1024, m=m)
                       for n in ("wq_b", "wkv", "wo_a", "wo_b") for m in (1, 8) for f in ("exact", "fast")},
        "upload": {f"depth{d}": {"s_per_batch": 0.017197224999996763, "h2d_gbps": 37.31581763919009} for d in (2, 4, 8)},
        "roofline": {"bound": "hbm", "achieved": 2795.0267424582003, "frac": 0.34937834280727503},
        "cpu_baseline": {"value": 44259.7429999978, "sample": "s" * 160, "all_cores": cores, "one_core": cores},
    }


def test_report_is_one_short_line_that_keeps_the_numbers():
    line = _line()
    assert len(json.dumps(line)) > 2 * bench.LINE_LIMIT  # what a default run measures
    text = bench.report(line)
    assert "\n" not in text and text.isascii() and len(text) <= bench.LINE_LIMIT
    got = json.loads(text)
    assert list(got) == list(line)
    for key, v in line.items():
        if not isinstance(v, dict):
            assert got[key] == v, key
    assert got["config"] == line["config"] and got["roofline"] == line["roofline"]
    assert got["fp8_linear"]["wo_b_m8_fast"]["us"] == 10.1
    assert got["k1"]["ms_range"] == [0.039506, 0.0404] and got["k1"]["eager_ms"] == 0.044  # the median
    assert "submission_covered" not in got["k1"]


def test_report_flags_an_uncovered_submission():
    line = {"k1": {"timing": _timing(0.04, covered=False)}, "k8": {"timing": {**_timing(0.1), "eager": _timing(0.1, covered=False)}}}
    got = json.loads(bench.report(line))
    assert got["k1"]["submission_covered"] is False and got["k8"]["submission_covered"] is False
