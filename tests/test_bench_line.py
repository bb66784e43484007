"""bench.py's printed line: one JSON object with the keys that a reader needs, short enough to be kept whole."""
import importlib.util
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_line_is_short_and_complete():
    """Every section measured, floats of full length, far more details than the line may hold."""
    bench = _bench()
    x = 123456.78901234567
    entry = bench.mfma_entry("gemm_tiles_kernel<swiglu>, one block per tile (gate/up projection + SwiGLU, as in the two-stream layer step), c4", 4 * 4096 * 1024 * 4096, x, x, x, x)
    expert = bench.hbm_entry("expert op (gather algorithm: expert_gather_kernel), config-5 shape (32768 tokens, hidden 2048, 262144 experts, top-32), ids uniform over the experts",
                             x, x, 10 ** 10, 10 ** 10, 10 ** 9, note="n" * 400)
    out = {"metric": "m" * 100, "value": x * 1e6, "unit": "tokens/s", "n_gpus": 1, "steps": 100, "warmup": 100, "ms_per_step": x, "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": "bf16", "data": "synthetic", "config": {"model": "c" * 200, "global_batch": 1, "seq_len": 4096, "parallelism": "one GPU"},
           "step_ms": {"median_single": x, "best_single": x, "repeats": 50, "protocol": "p" * 300}, "grad_enabled_forward": {"ms_per_step": x, "tokens_per_s": x, "note": "n" * 300},
           "roofline": entry, "roofline_expert": expert, "roofline_expert_hbm": expert, "kernels": [entry, expert] * 20, "ref_grid": [{"ms": x}] * 200, "mfma_probe": {"note": "n" * 500},
           "layer_c5": {"workload": "w" * 300, "ms_per_step": x, "tokens_per_s": x, "frac_of_mfma_peak": {"gate_up": x, "down": x, "router_projection": x}},
           "cpu_baseline": {"value": x, "unit": "tokens/s", "cores": 16, "kind": "port", "host_logical_cpus": 256, "cpu_model": "c" * 60, "sample": "s" * 200}}
    text = bench.headline(out)
    line = json.loads(text)
    assert "\n" not in text and len(text) <= bench.LINE_BYTES
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert key in line
    assert abs(line["value"] / out["value"] - 1) < 1e-6 and "kernels" not in line
    assert {"kernel", "bound", "achieved", "peak", "unit", "frac", "traffic"} <= set(line["roofline"])
    # a run of the timed steps alone prints what it has
    assert json.loads(bench.headline({"metric": "m", "value": x}))["value"] > 0
