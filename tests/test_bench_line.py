"""The benchmark's printed line stays short enough to be read from the end of an
output (under 11 KB with every section), and keeps the headline whole."""
import json

import bench


def test_printed_line_is_short_and_keeps_the_headline():
    figures = {k: 123.456789012345678 for k in ("tflops", "ms_per_call", "ms_median", "ms_min", "wall_s", "core_ms",
               "core_tflops", "max_rel_err", "mean_rel_err", "max_abs_err", "rms_abs_err", "max_err_over_bound_scale",
               "frac_of_fp32_vector_peak", "mfma_utilisation", "mfma_issue_frac", "roofline_peak", "frac_of_roofline")}
    forms = {f: dict(figures, core_kernel="split_nt_core") for f in bench.FORM_PEAK}
    line = {"metric": "m" * 80, "value": 417.7051234, "unit": "TFLOP/s", "n_gpus": 1, "steps": 20, "warmup": 5,
            "ms_per_step": 2.63231234, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "d" * 90, "data": "x" * 80, "config": {"workload": "w" * 500}, "forms": forms,
            "roofline": dict(figures), "target_3x_at_fp32_error": {f: dict(list(figures.items())[:5]) for f in forms},
            "config2_grid": {f"{n}_{t}_{f}": dict(figures) for n in (2048, 4096, 8192) for t in ("NN", "NT", "TN")
                             for f in ("fp32", "bf16x3", "fp16x3")},
            "config5_precision_ladder": forms}
    for name in bench.SECTIONS:
        line.setdefault(name, {str(i): dict(figures) for i in range(6)})
    whole, out = json.dumps(line), json.loads(json.dumps(bench.summary(line)))
    assert len(whole) > 20000 and len(json.dumps(out)) < 11000
    for k in line:
        if k not in bench.SECTIONS and k != "forms":
            assert out[k] == line[k]
    assert out["forms"]["fp16x3"]["tflops"] == 123.46 and len(out["config2_grid"]) == 27
    assert json.dumps(line) == whole   # the detail line is untouched
