"""bench.py's command line, as far as a machine without a GPU can check it."""

import pathlib
import subprocess
import sys

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_more_than_one_gpu_is_refused_with_a_message():
    done = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert done.returncode != 0
    assert "one GPU" in done.stderr and "--gpus 1" in done.stderr and done.stdout == ""


def test_the_default_workload_is_the_metrics_configuration():
    done = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--help"], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0
    for flag in ("--gpus", "--steps", "--warmup", "--config", "--bf16-operands"):
        assert flag in done.stdout


def test_the_lines_traffic_is_what_the_committed_summaries_hold():
    """`roofline.traffic` is parsed from the rocprofv3 summaries under profiles/: every workload has its rows there, the
    paired gate/up launches counted are the ones the same file's kernel trace times, and the figure in bytes is the
    summary's own scaled columns."""
    import re

    sys.path.insert(0, str(ROOT))
    import bench

    scales = bench.counter_scales()
    assert set(scales) == {"FETCH_SIZE", "WRITE_SIZE"} and all(0.5 <= factor <= 4.0 for factor in scales.values())
    for config in bench.ALL_CONFIGS:
        counted = bench.counted_kib(config)
        assert counted is not None and counted["FETCH_SIZE"] > 0 and counted["WRITE_SIZE"] > 0, config
        text = (ROOT / bench.COUNTED_FROM[config]).read_text()
        trace, traffic = text.split("2. HBM traffic", 1)
        assert f"--config {config} --only" in trace                      # the summary is of this workload's command
        paired = re.findall(r"^(dew::grouped_gemm_kernel<\d+, (?:1|3), [^>]*>(?: grid \d+)?)\s", traffic, re.M)
        assert paired and all(name in trace for name in paired), (config, paired)
        scaled = 0.0
        for line in traffic.splitlines():
            if any(line.startswith(name + " ") for name in paired):
                read, written = line.split()[-2:]
                scaled += float(read) + float(written)
        assert abs(bench.measured_traffic(config) - scaled) <= 2e-3 * scaled, (config, bench.measured_traffic(config), scaled)
    assert bench.counted_kib("c9") is None


def test_the_line_is_short_enough_to_be_kept_whole():
    """Every workload's figures in one line of at most 7 000 characters, whatever notes the record holds."""
    import json

    sys.path.insert(0, str(ROOT))
    import bench

    note, figure = "what a figure means, at length. " * 8, 1234.5678
    sustained = {"bf16_mfma_random_operands_tflops": figure, "plain_copy_gbs": figure, "read_stream_gbs": figure, "frac_of_sustained": 0.6711, "note": note}
    measured = {"value": figure, "unit": "TFLOP/s", "ms_per_step": 7.9532,
                "config": {"workload": "c4: T=8192 D=7168 F=2048 E=256 k=8 fp8_block weights, sigmoid router + shared expert", "routed_rows": 65536,
                           "experts_touched": 256, "shared_expert": "group #E of the routed launches",
                           "launch": "hip graph replay (the timed steps captured back to back as one graph)", "algorithmic_flops": 11544872091648.0},
                "roofline": {"bound": "mfma", "achieved": figure, "peak": 2500.0, "unit": "TFLOP/s", "peak_note": note, "frac": 0.5816, "frac_of_fp8_peak": 0.2908,
                             "frac_of_fp4_peak": 0.144, "hbm_view": {"algorithmic_bytes": 738197504.0, "gbs": figure, "frac_of_hbm_peak": 0.0585},
                             "executed": {"tflops": figure, "frac_of_fp8_peak": 0.5816, "note": note, "issue_time_frac": 0.58, "issue_time_note": note},
                             "traffic": 10**10, "traffic_source": note, "algorithmic": {"per_launch": 1924145348608.0, "unit": "flop"},
                             "sustained": sustained, "kernel": "grouped_gemm_kernel<paired gate/up + SwiGLU> on split rows (an instruction and its terms)",
                             "kernel_ms": 5.293},
                "router_logits": {"us": 59.7, "tflops_fp32": 17.99, "note": note},
                "min_topk_margin": {"value": 7.078051567077637e-06, "fp32_spacings": 475.0, "token": 1957, "note": note},
                "sample_parity": {"max_abs_over_max_ref": 0.00431, "elementwise": 0.012792, "identical_frac": 0.55503, "rows": 192, "experts": [4, 2, 3],
                                  "rows_note": note, "bar": 0.02}}
    whole = {"experts": "all 8 touched experts, every routed row", "routing_identical": True,
             "layer_output": {"max_abs_over_max_ref": 0.002475, "elementwise": 0.007752, "identical_frac": 0.99072}}
    baseline = {"value": 0.29041, "unit": "TFLOP/s", "cores": 16, "kind": "port", "sample": note, "gemm_only_tflops": 0.74487}
    configs = {name: dict(measured) for name in (*bench.ALL_CONFIGS, "c2_option_e2m3_second_term", "c2_option_two_e2m3_terms")}
    configs["c1"].update(cpu_baseline=baseline, sample_parity={**measured["sample_parity"], **whole})
    head = {"metric": "grouped-GEMM TFLOP/s & % MFMA peak (prefill); HBM GB/s & % peak (decode)", "n_gpus": 1, "steps": 20, "warmup": 5,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic"}
    printed = bench.line({**head, **measured, "cpu_baseline": baseline, "configs": configs}, "c2")
    assert len(printed) <= 7000 and "\n" not in printed
    kept = json.loads(printed)
    assert all(kept[key] == value for key, value in head.items()) and kept["value"] == figure and kept["ms_per_step"] == 7.9532
    assert kept["roofline"]["achieved"] == figure and kept["roofline"]["sustained"]["plain_copy_gbs"] == figure and kept["cpu_baseline"] == baseline
    assert set(kept["configs"]) == set(configs) - {"c2"}
    for part in kept["configs"].values():
        assert part["value"] == figure and part["roofline"]["frac"] == 0.5816 and part["sample_parity"]["elementwise"] == 0.012792
    assert "at length" not in json.dumps(kept["configs"]["c5"])
