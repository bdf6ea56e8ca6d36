"""bench.py's line for stdout, and --summarize-trace on a synthetic rocprofv3 CSV pair: only the
dispatches that start and end inside a "timed:<region>" range are counted,
per region occurrence, with the warm-up launches before the range left out."""
import csv
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _bench():
    spec = importlib.util.spec_from_file_location("bench_mod", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _write(path, rows):
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=list(rows[0]))
        w.writeheader()
        w.writerows(rows)


def test_summarize_trace_counts_timed_dispatches_only(tmp_path, capsys):
    us = 1000  # ns
    k = "void bmb::mfma_gemm_k<false, false, bmb::MfmaTile<256, 256, 32, 2, 4>, true, 0>(int, float)"
    kernels = [
        # warm-up, before the range
        {"Kernel_Name": k, "Start_Timestamp": 0, "End_Timestamp": 900 * us},
        # inside region "sgemm": 3 launches of 10, 20 and 30 us
        {"Kernel_Name": k, "Start_Timestamp": 1000 * us, "End_Timestamp": 1010 * us},
        {"Kernel_Name": k, "Start_Timestamp": 1020 * us, "End_Timestamp": 1040 * us},
        {"Kernel_Name": k, "Start_Timestamp": 1050 * us, "End_Timestamp": 1080 * us},
        # straddles the range's end: not counted
        {"Kernel_Name": k, "Start_Timestamp": 1090 * us, "End_Timestamp": 1200 * us},
        # second occurrence of the region: one launch
        {"Kernel_Name": "flash_fwd_h_k<64, 4, 1>(float*)", "Start_Timestamp": 2000 * us,
         "End_Timestamp": 2005 * us},
    ]
    markers = [
        {"Function": "timed:sgemm", "Start_Timestamp": 995 * us, "End_Timestamp": 1100 * us},
        {"Function": "untimed", "Start_Timestamp": 0, "End_Timestamp": 3000 * us},
        {"Function": "timed:sgemm", "Start_Timestamp": 1999 * us, "End_Timestamp": 2010 * us},
    ]
    _write(tmp_path / "run_kernel_trace.csv", kernels)
    _write(tmp_path / "run_marker_api_trace.csv", markers)
    _bench().summarize_trace(str(tmp_path))
    out = capsys.readouterr().out
    assert out.count("### region `sgemm`") == 2
    first, second = out.split("(occurrence 2)")
    row = [ln for ln in first.splitlines() if "mfma_gemm_k" in ln]
    assert len(row) == 1
    cells = [c.strip() for c in row[0].strip("|").split("|")]
    # kernel | calls | mean | median | min | max | total ms
    assert cells[0] == "`bmb::mfma_gemm_k<false, false, bmb::MfmaTile<256, 256, 32, 2, 4>, true, 0>`"
    assert cells[1:] == ["3", "20.0", "20.0", "10.0", "30.0", "0.060"]
    assert "flash_fwd_h_k<64, 4, 1>" in second and "mfma_gemm_k" not in second
    # a single region
    _bench().summarize_trace(str(tmp_path), "nothing")
    assert "### region" not in capsys.readouterr().out


def test_stdout_line_is_short_and_whole():
    """A full run's results (the sizes of every section) fit 7,500 characters,
    with the headline untouched, every section present and the verification
    reduced to its outcome."""
    import json
    rate, sizes = 123456.7, [str(n) for n in (512, 1000, 1024, 1536, 2048, 4096, 4097, 6144, 8192)]
    ids = ["id%d a_kernels_name" % i for i in range(1, 11)]
    ops = ("fwd_NT", "dX_NN", "dW_TN_beta1")
    telemetry = {"socket_power_w": 1402.9, "window_s": 1.0, "gfx_clk_mhz_per_xcd": [2254] * 8,
                 "gfx_clk_mhz_median": 2239, "gfx_clk_mhz_max_spec": 2400}
    step = {"metric": "m" * 80, "compute": "c" * 170, "value": 340841.2, "unit": "tokens/s",
            "ms_per_step": 24.035, "ms_best": 23.985, "steps": 20, "warmup": 3,
            "tflops_train_gpt_accounting": 293.16, "params": 124475904, "loss_first": 10.97762,
            "phase_ms": {"forward": 7.95, "backward": 15.51, "norm_clip_adamw": 0.73},
            "loss_last": 10.93974, "ln_V": 10.82491, "grad_norm_first": 2.82914,
            "device_telemetry_sustained": telemetry, "config": {"workload": "w" * 170}}
    line = {"metric": "m" * 70, "value": 144525.0, "unit": "GFLOP/s", "ms_per_step": 0.951,
            "config": {"workload": "w" * 130}, "vs_baseline": None, "data": "d" * 120,
            "roofline": {"traffic": 987654321, "peak_is": "p" * 100},
            "device_telemetry_sustained": telemetry,
            "config2_sweep_gflops": {i: {n: rate for n in sizes} for i in ids[:3]},
            "ladder_n4096": {i: {"gflops": rate, "pct_of_own_peak": 91.2, "peak_tflops": 157.3}
                             for i in ids},
            "config3_gpt_gemm_gflops": {
                s: {"shape": "8192x50304x768",
                    "bf16x3": dict({o: rate for o in ops}, pct_of_own_ceiling={o: 1.0 for o in ops}),
                    "fp32": dict({o: rate for o in ops}, pct_of_own_ceiling={o: 1.0 for o in ops}),
                    "vendor_fp32": {o: rate for o in ops}}
                for s in ("qkv", "attn_proj", "mlp_fc", "mlp_proj", "lm_head")},
            "flash": {"metric": "f" * 1700}, "cpu_baseline": {"sample": "s" * 370},
            "config5_gpt_train_step": step, "config5_gpt_train_step_fp32_gemm": dict(step),
            "verification": {"all_ok": True, "failed": [], "checks": {
                "check %d %s" % (i, "n" * 40): {"err": 1e-6 * i, "bound": 1e-4, "kind": "k" * 60,
                                                 "ok": True} for i in range(75)}}}
    text = _bench().summary_line(line)
    assert len(text) < 7500 and "\n" not in text
    out = json.loads(text)
    assert list(out) == list(line)
    for k in ("metric", "value", "unit", "ms_per_step", "config", "vs_baseline", "data", "roofline",
              "config2_sweep_gflops", "flash", "cpu_baseline"):
        assert out[k] == line[k]
    assert out["config3_gpt_gemm_gflops"]["qkv"]["bf16x3"] == {o: rate for o in ops}
    assert out["config5_gpt_train_step"]["value"] == 340841.2
    assert out["verification"]["checks"] == 75 and out["verification"]["all_ok"]
    assert out["verification"]["nearest_its_bound"]["name"].startswith("check 74")
