"""Benchmark of the OmniMoE forward hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--sections a,b,...]

Prints ONE JSON line of at most 4 KiB (a reader may keep only so much of a line); --details FILE
writes everything that was measured.  A step = one forward of the OmniMoE layer over one batch of
synthetic, HBM-resident input: the README shape (1 x 4096 tokens, hidden 1024, intermediate 4096,
4096 experts = 64 x 64 keys, top-16, bf16, train-mode BatchNorm), called config 4 below.
All timing uses HIP events recorded on the stream the kernels run on (torch's current stream;
the library enqueues there).

In the line:
  value          whole-layer tokens/s over the K timed steps (one event pair around all K)
  step_ms        the same step timed one at a time with a freshly cloned input per repeat, as the
                 reference's harness does (tests/testing.py:152-212): median and best
  grad_enabled_forward   the same call with autograd recording
  roofline       the kernel that takes the largest share of a step (gate/up MFMA GEMM); its
                 duration is the average over back-to-back launches between one event pair, so
                 that it matches what a kernel trace shows
  roofline_expert        the expert op on benchmark config 3 (16384 tokens), whose 16 MiB tables are
                         cache-resident: fraction of HBM peak from the bytes that really cross the fabric
  roofline_expert_hbm    the expert op at benchmark config 5's shape (2 GiB tables): HBM-resident, so
                         algorithmic bytes are HBM bytes
  layer_c5       the whole layer at benchmark config 5 (32768 tokens, hidden 2048, intermediate 8192, 262144
                 experts, top-32, Zipf-skewed keys): step time, tokens/s and its three MFMA GEMMs
  cpu_baseline   the oracle (the reference's PyTorch layer restated with torch CPU ops) on the
                 host cores, same workload
Only among the details:
  kernels        per-launch figures for every stage, with what each counts and where its byte figures come from
  mfma_probe     what the matrix cores sustain on register operands
  ref_grid       the shapes of the reference's own operator benchmarks (tests/test_router.py:103-110,
                 tests/test_expert.py:181-187, tests/test_mlp.py:144-150), each beside the same operator
                 composed from torch library ops on this GPU

Sections (default: all): layer, kernels, expert_c3, expert_c5, layer_c5, ref_grid, probe, train, cpu.
"""
import argparse
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for p in (os.path.join(ROOT, "omni-moe_amd"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)

HBM_PEAK_GBS = 8000.0           # MI355X HBM3E, published
MFMA_BF16_PEAK_TFLOPS = 2500.0  # MI355X dense bf16, published
# Bytes that cross the fabric per launch (FETCH_SIZE + WRITE_SIZE of rocprofv3 --pmc, each scaled by a plain copy of
# known size); counters cannot be read in-process, so these are the figures of the committed summaries named here.
TRAFFIC_SOURCE = ("profiles/bench_layer_c4_hbm_counters.txt, profiles/expert_c5_hbm_counters.txt; measured on the kernels as of the commit "
                  "'Split expert passes: no ragged kernels for groups of four lanes, which no cut produces', the expert backward's as of "
                  "'Expert weight pass: short segments stay with the wave that begins them, rows of the gradients stored past the L2' -- a "
                  "later change to a kernel's memory access pattern needs a new counter run")
TRAFFIC_BYTES = {"expert_c3": 132.4e6, "expert_c4": 58.3e6, "expert_gather_c3": 899.2e6, "gateup_c4": 134.4e6, "down_c4": 117.6e6,
                 "down_plain_c4": 109.2e6, "schedule_c3": 12.4e6, "expert_segment_c3": 927.1e6, "expert_bwd_c3": 1325.5e6,
                 "expert_c5_routed": 1030.3e6, "expert_c5_routed_split": 731.5e6, "expert_c5_uniform": 8846.5e6}
SECTIONS = ("layer", "kernels", "expert_c3", "expert_c5", "layer_c5", "ref_grid", "probe", "train", "cpu")


def expert_alg_bytes(T, H, k, s=2):
    """Gather model: per token the x row, k up rows, k down rows, the y row, k ids and k gates."""
    return T * ((2 * k + 2) * H * s + k * (4 + s))


def expert_min_bytes(T, H, N, k, s=2):
    """Compulsory traffic: x and y once, every table row that is used at least once (at most the tables), ids and gates."""
    P = T * k
    return 2 * T * H * s + min(2 * N * H * s, 2 * P * H * s) + P * (4 + s)


def expert_bwd_alg_bytes(T, H, N, k, s=2):
    """Backward of the expert op.  Token pass: x, dy and dx rows, k up rows, k down rows, k ids, gates and dgates,
    k fp32 (ds, coef) pairs out.  Weight pass: per pair the x and dy rows, its two fp32 coefficients, pair id and token
    id; the dU and dV tables out.  Plus the schedule."""
    P = T * k
    token_pass = T * (2 * k + 3) * H * s + P * (4 + 2 * s + 8)
    weight_pass = P * (2 * H * s + 16) + 2 * N * H * s
    return token_pass + weight_pass + P * 14 + 8 * (N + 1)


def time_launches(torch, fn, n=40, reps=5, warmup=5):
    """Milliseconds per launch of fn: n launches back to back between one event pair (so that host gaps and
    event latency do not count), repeated; returns (median, best)."""
    for _ in range(warmup):
        fn()
    out = []
    for _ in range(reps):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        s.record()
        for _ in range(n):
            fn()
        e.record()
        torch.cuda.synchronize()
        out.append(s.elapsed_time(e) / n)
    return statistics.median(out), min(out)


def router_stage_call(torch, _lib, layer, x, training):
    """omni_router_fwd on the layer's router parameters with outputs and workspace allocated once, the way the layer's
    single library call drives it (the Python operator allocates its outputs per call, which at a 20 us stage is most
    of what a loop over it measures).  Returns a zero-argument callable that enqueues one stage."""
    lib = _lib.load()
    T, H = x.shape
    r, k = layer.num_expert_sqrt, layer.top_k
    nx, ny = layer._router_norms()
    dt, sdt = _lib.DTYPE_CODE[x.dtype], _lib.DTYPE_CODE[nx.running_mean.dtype]
    gates = torch.empty(T, k, dtype=x.dtype, device=x.device)
    ids = torch.empty(T, k, dtype=torch.int32, device=x.device)
    ws = torch.empty(lib.omni_router_workspace_bytes(T, r, dt), dtype=torch.uint8, device=x.device)
    wx, wy = layer.router_gate_x.weight, layer.router_gate_y.weight
    keep = (gates, ids, ws)

    def call():
        _lib.check(lib.omni_router_fwd(x.data_ptr(), wx.data_ptr(), wy.data_ptr(), nx.running_mean.data_ptr(), nx.running_var.data_ptr(),
                                       nx.num_batches_tracked.data_ptr(), ny.running_mean.data_ptr(), ny.running_var.data_ptr(),
                                       ny.num_batches_tracked.data_ptr(), int(training), float(nx.momentum), float(nx.eps),
                                       gates.data_ptr(), ids.data_ptr(), None, T, H, r, k, dt, sdt, ws.data_ptr(), _lib.stream_ptr()),
                   "omni_router_fwd")
    call.keep = keep
    return call


def hbm_entry(name, ms, best, alg_bytes, traffic=None, min_bytes=None, resident_in_hbm=False, note=None):
    """Bandwidth-bound kernel.  `achieved`/`frac` use the bytes that really move: measured fabric traffic where a
    counter run exists, algorithmic bytes where the working set is HBM-resident; cache-served algorithmic bytes are
    reported as a rate of their own, never as a fraction of HBM peak."""
    d = {"kernel": name, "bound": "hbm", "peak": HBM_PEAK_GBS, "unit": "GB/s", "kernel_ms": ms, "kernel_ms_best": best,
         "algorithmic_bytes": alg_bytes, "algorithmic_rate_GBs": alg_bytes / (ms * 1e-3) / 1e9, "traffic": traffic}
    moved = alg_bytes if resident_in_hbm else traffic
    if moved is not None:
        d["achieved"] = moved / (ms * 1e-3) / 1e9
        d["frac"] = d["achieved"] / HBM_PEAK_GBS
        d["achieved_from"] = "algorithmic bytes (working set is HBM-resident)" if resident_in_hbm else "measured fabric traffic"
    else:
        d["achieved"] = d["frac"] = None
    if min_bytes is not None:
        d["compulsory_bytes"] = min_bytes
        d["frac_compulsory"] = min_bytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS
    if note:
        d["note"] = note
    return d


def mfma_entry(name, flops, ms, best, traffic=None, sustained=None):
    a = flops / (ms * 1e-3) / 1e12
    d = {"kernel": name, "bound": "mfma", "achieved": a, "peak": MFMA_BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
         "frac": a / MFMA_BF16_PEAK_TFLOPS, "traffic": traffic, "algorithmic_flops": flops, "kernel_ms": ms, "kernel_ms_best": best}
    if sustained:
        d["sustained_mfma_rate"] = sustained
        d["frac_of_sustained"] = a / sustained
    return d


#: What the printed line holds: keys of the full result, each whole (None) or the named parts of it.
LINE = {**{k: None for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype",
                             "data", "config")},
        "step_ms": ("median_single", "best_single", "repeats"), "grad_enabled_forward": ("ms_per_step", "tokens_per_s"),
        **{k: ("kernel", "bound", "achieved", "peak", "unit", "frac", "kernel_ms", "traffic", "frac_of_sustained", "frac_compulsory", "library_gemm_same_flops_ms")
           for k in ("roofline", "roofline_expert", "roofline_expert_hbm")},
        "layer_c5": ("ms_per_step", "tokens_per_s", "frac_of_mfma_peak"), "cpu_baseline": None}
LINE_BYTES = 4096


def short(v):
    """Floats to seven figures: more than a timing has, and half the text."""
    if isinstance(v, dict):
        return {k: short(x) for k, x in v.items()}
    return float(f"{v:.7g}") if isinstance(v, float) else v


def headline(out):
    """The printed line: the entries of LINE that were measured."""
    line = {}
    for key, parts in LINE.items():
        if key in out:
            line[key] = short(out[key] if parts is None else {p: out[key][p] for p in parts if p in out[key]})
    text = json.dumps(line)
    assert len(text) <= LINE_BYTES, len(text)
    return text


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=100,
                    help="untimed steps; the first ~100 steps after the GPU has idled run about 7 %% slower (clocks ramp up)")
    ap.add_argument("--sections", default=",".join(SECTIONS), help="comma-separated subset of: " + ", ".join(SECTIONS))
    ap.add_argument("--details", metavar="FILE", help="also write every figure measured to FILE, as JSON")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-kernels", action="store_true", help="only the layer steps (profiling runs)")
    ap.add_argument("--calibration-copy", action="store_true",
                    help="also run a plain 256 MiB device copy 3 times (known traffic, to scale HBM byte counters)")
    a = ap.parse_args()
    if a.gpus != 1:
        sys.exit("bench.py: this build runs on ONE GPU; --gpus must be 1 (no multi-GPU path exists)")
    sections = set(s for s in a.sections.split(",") if s)
    unknown = sections - set(SECTIONS)
    if unknown:
        sys.exit(f"bench.py: unknown sections {sorted(unknown)}")
    if a.no_cpu_baseline:
        sections.discard("cpu")
    if a.no_kernels:
        sections &= {"layer", "cpu"}

    import torch
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    from omni_moe.ops import hip
    from omni_moe.ops.hip import _lib
    from oracle import omni_oracle as oracle          # checker + cpu_baseline leg only

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    torch.set_grad_enabled(False)          # forward path: the module then issues its single fused library call

    # ---------------- benchmark config 4: README-shape full layer
    T, H, I, N, k, seed = 4096, 1024, 4096, 4096, 16, 3
    x, w = oracle.make_layer_inputs(seed, T, H, I, N)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    layer.load_state_dict({"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
                           "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
                           "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}, strict=False)
    layer = layer.to(device=dev, dtype=torch.bfloat16)          # module default: training mode (batch-stat BN)
    dx = x.to(dev)

    out = {
        "metric": "OmniMoE fwd tokens/sec @h1024,N4096,k16 (1 GPU); expert kernel HBM GB/s %peak",
        "value": None, "unit": "tokens/s", "n_gpus": 1, "steps": a.steps, "warmup": a.warmup,
        "ms_per_step": None, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"model": f"OmniMoE layer forward: hidden {H}, intermediate {I}, {N} experts (64x64 keys), top-{k}, silu, train-mode BatchNorm, seed {seed}",
                   "global_batch": 1, "seq_len": T, "parallelism": "one GPU"},
    }

    for _ in range(a.warmup):
        y = layer(dx)
    torch.cuda.synchronize()
    s_all, e_all = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    s_all.record()
    for _ in range(a.steps):
        y = layer(dx)
    e_all.record()
    torch.cuda.synchronize()
    out["wall_s_timed_region"] = time.perf_counter() - t0
    out["ms_per_step"] = s_all.elapsed_time(e_all) / a.steps
    out["value"] = T / (out["ms_per_step"] * 1e-3)

    if "layer" in sections:
        # the reference's protocol (tests/testing.py:152-212): a fresh clone of the input per repeat, synchronise, time one call
        reps = max(20, min(a.steps, 50))
        per = []
        for _ in range(reps):
            xi = dx.clone()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats(dev)
            s.record()
            layer(xi)
            e.record()
            torch.cuda.synchronize()
            per.append(s.elapsed_time(e))
        out["step_ms"] = {"mean_back_to_back": out["ms_per_step"], "median_single": statistics.median(per), "best_single": min(per),
                          "repeats": reps, "peak_memory_MiB": torch.cuda.max_memory_allocated(dev) / 2 ** 20,
                          "protocol": "single: fresh cloned input, synchronise, events around one call (reference tests/testing.py:152-212); "
                                      "back_to_back: the K timed steps between one event pair"}
        # the layer exactly as the reference's README calls it: grad enabled, parameters requiring grad
        # (one differentiable node, not the single fused call)
        with torch.enable_grad():
            g_med, g_best = time_launches(torch, lambda: layer(dx), n=20, reps=5, warmup=3)
        out["grad_enabled_forward"] = {"ms_per_step": g_med, "ms_per_step_best": g_best, "tokens_per_s": T / (g_med * 1e-3),
                                       "note": "moe(x) with autograd recording (README quick start), as one differentiable node; the gate/up GEMM "
                                               "also stores gate and up for the backward pass"}

        # correctness spot check against the oracle (outside the timed region): eval mode on both
        # sides so that the repeated train-mode steps above do not matter
        layer.eval()
        sub = 256
        y_sub = layer(dx[:, :sub]).float().cpu()
        bx, by = oracle.BNState.fresh(layer.num_expert_sqrt), oracle.BNState.fresh(layer.num_expert_sqrt)
        bx.running_mean, bx.running_var = layer.router_norm_x.running_mean.float().cpu(), layer.router_norm_x.running_var.float().cpu()
        by.running_mean, by.running_var = layer.router_norm_y.running_mean.float().cpu(), layer.router_norm_y.running_var.float().cpu()
        want, _, _ = oracle.moe_forward(x[:, :sub], w, bx, by, k, training=False)
        torch.testing.assert_close(y_sub, want.float(), rtol=2e-2, atol=2e-2)
        layer.train()

    if a.calibration_copy:
        src = torch.empty(256 << 20, dtype=torch.uint8, device=dev).fill_(1)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    kernels = []
    sustained = sustained32 = None
    if "probe" in sections:
        # matrix-core rate with nothing else going on, on 8 KiB of the real activations: the clock that the board
        # sustains under its power limit depends on the operand bits, so this is the ceiling a GEMM on this data has
        lib = _lib.load()
        blocks, iters = 1024, 2048
        sink = torch.empty(blocks * 512, device=dev, dtype=torch.float32)
        ops = dx.view(-1)[:4096].contiguous()
        zeros = torch.zeros_like(ops)

        def probe(fn, data, flop):
            ms, _ = time_launches(torch, lambda: _lib.check(fn(data.data_ptr(), sink.data_ptr(), blocks, iters, _lib.stream_ptr()), "omni_probe_mfma"),
                                  n=3, reps=3, warmup=1)
            return flop / (ms * 1e-3) / 1e12
        flop32, flop16 = blocks * 4 * iters * 16 * 32768, blocks * 8 * iters * 32 * 16384
        sustained32 = probe(lib.omni_probe_mfma, ops, flop32)
        sustained = probe(lib.omni_probe_mfma16, ops, flop16)       # the instruction of the 256 x 256 GEMM kernel
        out["mfma_probe"] = {"sustained_TFLOPs_on_activations": sustained, "sustained_TFLOPs_on_zeros": probe(lib.omni_probe_mfma16, zeros, flop16),
                             "sustained_TFLOPs_on_activations_32x32x16": sustained32,
                             "sustained_TFLOPs_on_zeros_32x32x16": probe(lib.omni_probe_mfma, zeros, flop32),
                             "published_peak_TFLOPs": MFMA_BF16_PEAK_TFLOPS,
                             "note": "v_mfma_f32_16x16x32_bf16 (8 waves per CU) and v_mfma_f32_32x32x16_bf16 (4 waves per CU) from registers only, "
                                     "no memory traffic: what the matrix cores sustain under the board's power limit; with realistic operand "
                                     "bits it is well below the published peak, and the 16x16x32 instruction sustains more"}

    if "kernels" in sections:
        xf = dx.view(-1, H)
        gates, ids = layer.route(xf)
        e_out = hip.hip_omni_expert_func(xf, layer.up_embed.weight, layer.down_embed.weight, gates, ids)
        h = hip.hip_swiglu_linear_func(xf, layer.gate_proj.weight, layer.up_proj.weight)
        y0 = hip.hip_linear_func(h, layer.down_proj.weight)
        r = layer.num_expert_sqrt
        # the gate/up projection as the two-stream layer step runs it (one block per tile: 512 blocks that leave room for the side branch as they retire) ...
        m, b = time_launches(torch, lambda: hip.hip_swiglu_linear_func(xf, layer.gate_proj.weight, layer.up_proj.weight, shared=True))
        kernels.append(mfma_entry("gemm_tiles_kernel<swiglu>, one block per tile (gate/up projection + SwiGLU, as in the two-stream layer step), c4", 4 * T * H * I, m, b, TRAFFIC_BYTES["gateup_c4"], sustained))
        # ... and as every caller gets it that has the GPU to itself (operator calls, the one-stream layer): one block per CU streaming through its tiles
        m_s, b_s = time_launches(torch, lambda: hip.hip_swiglu_linear_func(xf, layer.gate_proj.weight, layer.up_proj.weight))
        kernels[-1]["streaming_form_alone_ms"] = m_s
        kernels[-1]["streaming_form_alone_ms_best"] = b_s
        kernels[-1]["streaming_form_frac"] = 4 * T * H * I / (m_s * 1e-3) / 1e12 / MFMA_BF16_PEAK_TFLOPS
        # for orientation: the vendor library (torch.matmul) on the same operands, without the SwiGLU (one GEMM over [Wg; Wu])
        wcat = torch.cat([layer.gate_proj.weight, layer.up_proj.weight], 0)
        m_lib, b_lib = time_launches(torch, lambda: torch.matmul(xf, wcat.t()))
        kernels[-1]["library_gemm_same_flops_ms"] = m_lib
        m_lib, b_lib = time_launches(torch, lambda: torch.matmul(h, layer.down_proj.weight.t()))
        del wcat
        m, b = time_launches(torch, lambda: hip.hip_linear_func(h, layer.down_proj.weight, e_out))
        kernels.append(mfma_entry("gemm_tiles_kernel<residual> (down projection + experts add), c4", 2 * T * H * I, m, b, TRAFFIC_BYTES["down_c4"], sustained))
        m, b = time_launches(torch, lambda: hip.hip_linear_func(h, layer.down_proj.weight))
        kernels.append(mfma_entry("gemm_tiles_kernel<plain> (down projection alone, as on the two-stream path), c4", 2 * T * H * I, m, b, TRAFFIC_BYTES["down_plain_c4"], sustained))
        kernels[-1]["library_gemm_same_flops_ms"] = m_lib
        m, b = time_launches(torch, lambda: hip.hip_add_inplace_func(y0, e_out))
        kernels.append(hbm_entry("add_inplace_kernel (join of the two branches), c4", m, b, 3 * T * H * 2, resident_in_hbm=False,
                                 note="24 MiB that the caches hold between launches"))
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(xf, layer.up_embed.weight, layer.down_embed.weight, gates, ids))
        kernels.append(hbm_entry("expert op (split algorithm: expert_split_dots_kernel + expert_split_accumulate_kernel), c4", m, b,
                                 expert_alg_bytes(T, H, k), TRAFFIC_BYTES["expert_c4"], expert_min_bytes(T, H, N, k)))
        m, b = time_launches(torch, router_stage_call(torch, _lib, layer, xf, True))
        m_e, b_e = time_launches(torch, router_stage_call(torch, _lib, layer, xf, False))
        m_op, _ = time_launches(torch, lambda: layer.route(xf))
        kernels.append({"kernel": "router stage (projection GEMM with BN statistics epilogue + BN finalize + select), c4", "kernel_ms": m,
                        "kernel_ms_best": b, "eval_mode_ms": m_e, "eval_mode_ms_best": b_e, "through_python_operator_ms": m_op,
                        "timed": "omni_router_fwd through the C ABI with outputs and workspace allocated once, as the layer call runs it; "
                                 "through_python_operator_ms is a loop over layer.route(x), which allocates per call and is host-bound",
                        "algorithmic_flops": 4 * T * H * r, "algorithmic_bytes": (T * H + 2 * r * H + T * k * 3) * 2,
                        "note": "1.07 GFLOP over 9.7 MB: bounded by launch and memory latency, not by a roofline; two dependent launches: in training the selecting "
                                "blocks merge the batch statistics, in eval they read the running ones"})
        out["roofline"] = kernels[0]

    if "expert_c3" in sections:
        # expert op at benchmark config 3, the shape its bandwidth target is quoted on
        T3 = 16384
        x3c, up3c, down3c, g3c, i3c = oracle.make_expert_inputs(2, T3, H, N, k)
        x3, up3, down3, g3, i3 = (t.to(dev) for t in (x3c, up3c, down3c, g3c, i3c))
        y3 = hip.hip_omni_expert_func(x3, up3, down3, g3, i3)
        sub = 512                                      # checked against the oracle on a token subset, outside any timed region
        want3 = oracle.expert_forward(x3c[:sub], up3c, down3c, g3c[:sub], i3c[:sub])
        torch.testing.assert_close(y3[:sub].float().cpu(), want3.float(), rtol=2e-2, atol=2e-2)
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(x3, up3, down3, g3, i3))
        e3 = hbm_entry("expert op (split algorithm: expert_split_dots_kernel + expert_split_accumulate_kernel), c3 (T=16384)", m, b,
                       expert_alg_bytes(T3, H, k), TRAFFIC_BYTES["expert_c3"], expert_min_bytes(T3, H, N, k),
                       note="the 16 MiB tables are cache-resident (each XCD's L2 holds the quarter of them its blocks use): the kernel is bound "
                            "on the chip (L2 hits), so the fraction of HBM peak counts only the bytes that cross the fabric")
        kernels.append(e3)
        out["roofline_expert"] = e3
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(x3, up3, down3, g3, i3, algo="gather"))
        kernels.append(hbm_entry("expert op, gather algorithm (expert_gather_kernel), c3", m, b, expert_alg_bytes(T3, H, k),
                                 TRAFFIC_BYTES["expert_gather_c3"], expert_min_bytes(T3, H, N, k),
                                 note="for comparison: whole rows per wave, three quarters of them fetched over the fabric"))
        m, b = time_launches(torch, lambda: hip.hip_omni_schedule_func(i3, N))
        kernels.append(hbm_entry("schedule (stable counting sort of the pairs by expert: sort_count_kernel + sort_scatter_kernel), c3", m, b,
                                 T3 * k * 12 + 4 * (N + 1), TRAFFIC_BYTES["schedule_c3"],
                                 note="ids in, pair ids + token ids + offsets out; writes equal the algorithmic 2.1 MB (every output line goes through one L2), the ids are fetched by all 8 XCDs"))
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(x3, up3, down3, g3, i3, algo="segment"))
        kernels.append(hbm_entry("expert op, expert-centric 'segment' algorithm (schedule + scores pass + token pass), c3", m, b,
                                 expert_alg_bytes(T3, H, k), TRAFFIC_BYTES["expert_segment_c3"], expert_min_bytes(T3, H, N, k),
                                 note="for comparison; same results as the gather algorithm"))
        # the reference's group regime (omni_scheduler.py:58: tokens x k / experts > 256): same tokens, 256 experts; the
        # dense algorithm by name (two MFMA GEMMs over all experts), timed beside the gather algorithm on the same inputs
        Ng = 256
        xg_c, upg_c, downg_c, gg_c, ig_c = oracle.make_expert_inputs(2, T3, H, Ng, k)
        xg, upg, downg, gg, ig = (t.to(dev) for t in (xg_c, upg_c, downg_c, gg_c, ig_c))
        yg = hip.hip_omni_expert_func(xg, upg, downg, gg, ig, algo="dense")
        wantg = oracle.expert_forward(xg_c[:sub], upg_c, downg_c, gg_c[:sub], ig_c[:sub])
        torch.testing.assert_close(yg[:sub].float().cpu(), wantg.float(), rtol=2e-2, atol=2e-2)
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(xg, upg, downg, gg, ig, algo="dense"))
        dense = mfma_entry("expert op, dense algorithm (gate rows + transpose + two MFMA GEMMs), group regime: 16384 tokens, 256 experts, top-16",
                           2 * T3 * H * Ng + 2 * T3 * H * 2 * Ng, m, b, None, None)
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(xg, upg, downg, gg, ig, algo="gather"))
        dense["gather_algorithm_ms"] = m
        dense["note"] = ("1024 pairs per expert: every token meets every expert in a [T,N] product; the flop count is the dense one "
                         "(6 T H N), the selected pairs alone would be 4 T k H")
        kernels.append(dense)
        del xg, upg, downg, gg, ig, yg
        if "train" in sections:
            # training path (not part of the forward metric): backward of the expert op at the same shape
            dy3 = x3 * 0.5
            m, b = time_launches(torch, lambda: hip.hip_omni_expert_bwd_func(dy3, x3, up3, down3, g3, i3), n=10)
            kernels.append(hbm_entry("expert op backward (schedule + token pass + weight pass), c3", m, b, expert_bwd_alg_bytes(T3, H, N, k),
                                     TRAFFIC_BYTES["expert_bwd_c3"], note="x, dy (32 MiB each) and the tables are cache-resident"))
        del x3, up3, down3, g3, i3, y3

    if "expert_c5" in sections or "layer_c5" in sections:
        # benchmark config 5: 32768 tokens, hidden 2048, intermediate 8192, 262144 experts (512 x 512 keys), top-32; 2 GiB of
        # expert tables, so every selected row that is not reused comes from HBM.  Key popularity ~ Zipf(1.1) through
        # eval-mode BatchNorm buffers (running_mean = 1.1 ln(1+i), running_var = 1 - eps: a per-key bias on the normalised
        # logits; the reference's router has no bias of its own, omni_moe.py:47-52).  Weights are drawn on the device.
        T5, H5, I5, N5, k5, r5 = 32768, 2048, 8192, 262144, 32, 512
        g = torch.Generator(device=dev).manual_seed(4)
        draw = lambda *shape, std: torch.empty(*shape, device=dev, dtype=torch.bfloat16).normal_(0, std, generator=g)
        x5 = draw(T5, H5, std=1.0)
        up5, down5 = draw(N5, H5, std=0.02), draw(N5, H5, std=0.02)
        wx5, wy5 = draw(r5, H5, std=0.02), draw(r5, H5, std=0.02)
        rm = (1.1 * torch.log1p(torch.arange(r5, dtype=torch.float32))).to(device=dev, dtype=torch.bfloat16)
        rv = torch.full((r5,), 1.0 - 1e-5, device=dev, dtype=torch.bfloat16)
        g5, i5 = hip.hip_omni_router_fwd_func(x5, wx5, wy5, rm, rv, None, rm.clone(), rv.clone(), None, k5, training=False)
        sub = 64                                          # tokens checked against the oracle, over the table rows they select

        def expert_want5(gates, ids):
            rows, inv = torch.unique(ids[:sub].long(), return_inverse=True)
            return oracle.expert_forward(x5[:sub].cpu(), up5[rows].cpu(), down5[rows].cpu(), gates[:sub].cpu(), inv.cpu().to(torch.int32))

        def check5(y, gates, ids):
            torch.testing.assert_close(y[:sub].float().cpu(), expert_want5(gates, ids).float(), rtol=2e-2, atol=2e-2)

    if "expert_c5" in sections:
        y5 = hip.hip_omni_expert_func(x5, up5, down5, g5, i5)
        check5(y5, g5, i5)
        used = torch.unique(i5).numel()
        counts = torch.bincount(i5.flatten().long(), minlength=N5)
        alg5 = expert_alg_bytes(T5, H5, k5)
        min5 = 2 * T5 * H5 * 2 + 2 * used * H5 * 2 + T5 * k5 * 6
        skew = (f"the skewed router selects only {used} distinct experts (the most popular takes {int(counts.max())} of the {T5 * k5} pairs): "
                "their rows stay in the caches, so few of the algorithmic bytes cross the fabric")
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(x5, up5, down5, g5, i5, algo="gather"), n=10, reps=5, warmup=2)
        kernels.append(hbm_entry("expert op (gather algorithm: expert_gather_kernel), config-5 shape (32768 tokens, hidden 2048, 262144 experts, top-32), "
                                 "ids from the config-5 router (key popularity ~ Zipf(1.1))", m, b, alg5, TRAFFIC_BYTES["expert_c5_routed"], min5, note=skew))
        # the hidden-split algorithm on the same ids: which one wins depends on how many distinct rows are live, which the
        # table size alone (all AUTO can see without a host sync) does not tell
        ys = hip.hip_omni_expert_func(x5, up5, down5, g5, i5, algo="split")
        check5(ys, g5, i5)
        m_s, b_s = time_launches(torch, lambda: hip.hip_omni_expert_func(x5, up5, down5, g5, i5, algo="split"), n=10, reps=5, warmup=2)
        kernels.append(hbm_entry("expert op (split algorithm: expert_split_dots_kernel + expert_split_accumulate_kernel), config-5 shape, "
                                 "ids from the config-5 router (key popularity ~ Zipf(1.1))", m_s, b_s, alg5, TRAFFIC_BYTES.get("expert_c5_routed_split"), min5,
                                 note="same inputs as the entry above, algo='split' by name (OmniMoE.expert_algo = 'split'): the live rows' column slices fit the XCDs' L2s"))
        m_a, b_a = time_launches(torch, lambda: hip.hip_omni_expert_func(x5, up5, down5, g5, i5), n=10, reps=5, warmup=2)
        out["expert_c5_routed"] = {"gather_ms": m, "split_ms": m_s, "auto_ms": m_a, "distinct_experts": used, "max_pairs_per_expert": int(counts.max()),
                                   "note": "AUTO decides from the sizes alone (512-byte row slices and a million pairs: split); the layer takes a hint (OmniMoE.expert_algo) where the caller knows better"}
        # the same shape with ids spread evenly (32 distinct experts per token, uniform over all 262144): every selected
        # row comes from HBM, so algorithmic bytes are HBM bytes -- the case that shows the kernel against the HBM roofline
        iu = torch.randint(0, N5 // k5, (T5, k5), device=dev, generator=g, dtype=torch.int32) * k5 + torch.arange(k5, device=dev, dtype=torch.int32)
        yu = hip.hip_omni_expert_func(x5, up5, down5, g5, iu, algo="gather")
        check5(yu, g5, iu)
        m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(x5, up5, down5, g5, iu, algo="gather"), n=10, reps=5, warmup=2)
        m_us, _ = time_launches(torch, lambda: hip.hip_omni_expert_func(x5, up5, down5, g5, iu, algo="split"), n=10, reps=5, warmup=2)
        e5 = hbm_entry("expert op (gather algorithm: expert_gather_kernel), config-5 shape (32768 tokens, hidden 2048, 262144 experts, top-32), ids uniform over the experts",
                       m, b, alg5, TRAFFIC_BYTES["expert_c5_uniform"], 2 * T5 * H5 * 2 + 2 * torch.unique(iu).numel() * H5 * 2 + T5 * k5 * 6, resident_in_hbm=True,
                       note="2 GiB of tables, no reuse to speak of: the rocprofv3 byte counters of this launch read the algorithmic bytes (profiles/expert_c5_hbm_counters.txt)")
        e5["split_algorithm_same_ids_ms"] = m_us            # what AUTO runs at this shape; no byte counters were taken for it
        kernels.append(e5)
        out["roofline_expert_hbm"] = e5
        del y5, ys, iu, yu

    if "layer_c5" in sections:
        layer5 = OmniMoE(OmniMoEConfig(H5, I5, "silu", N5, k5))
        layer5 = layer5.to(device=dev, dtype=torch.bfloat16).eval()
        with torch.no_grad():
            layer5.gate_proj.weight.copy_(draw(I5, H5, std=0.02)); layer5.up_proj.weight.copy_(draw(I5, H5, std=0.02))
            layer5.down_proj.weight.copy_(draw(H5, I5, std=0.02))
            layer5.router_gate_x.weight.copy_(wx5); layer5.router_gate_y.weight.copy_(wy5)
            for bn in (layer5.router_norm_x, layer5.router_norm_y):
                bn.running_mean.copy_(rm); bn.running_var.copy_(rv)
        # the 2 GiB tables are the ones drawn above: the module's parameters alias them (no second copy in HBM)
        layer5.up_embed.weight.data, layer5.down_embed.weight.data = up5, down5
        per_algo = {}
        for algo in ("auto", "gather"):                 # AUTO takes the split algorithm at this shape
            layer5.expert_algo = algo
            y5l = layer5(x5.view(8, T5 // 8, H5)).view(T5, H5)
            # oracle on a token subset (eval mode is token-independent): router ids, then experts over the selected rows + MLP
            bx = oracle.BNState(rm.float().cpu(), rv.float().cpu(), torch.zeros((), dtype=torch.long))
            by = oracle.BNState(rm.float().cpu(), rv.float().cpu(), torch.zeros((), dtype=torch.long))
            wg_, wi_, _ = oracle.router_forward(x5[:sub].cpu(), wx5.cpu(), wy5.cpu(), bx, by, k5, False)
            agree = (i5[:sub].cpu().sort(-1).values == wi_.sort(-1).values).float().mean().item()
            assert agree >= 0.99, agree
            want5 = (oracle.mlp_forward(x5[:sub].cpu(), layer5.gate_proj.weight.cpu(), layer5.up_proj.weight.cpu(), layer5.down_proj.weight.cpu()).float()
                     + expert_want5(g5, i5).float())
            torch.testing.assert_close(y5l[:sub].float().cpu(), want5, rtol=2e-2, atol=2e-2)
            m, b = time_launches(torch, lambda: layer5(x5.view(8, T5 // 8, H5)), n=5, reps=5, warmup=2)
            per_algo[algo] = {"ms_per_step": m, "ms_per_step_best": b, "tokens_per_s": T5 / (m * 1e-3)}
        layer5.expert_algo = "auto"
        # the module's default at this size is one stream (OmniMoE.overlap_max_work); the two-stream schedule beside it
        layer5.overlap_max_work = 2 ** 62
        m2, b2 = time_launches(torch, lambda: layer5(x5.view(8, T5 // 8, H5)), n=5, reps=5, warmup=2)
        del layer5.overlap_max_work
        xf5 = x5
        m_gu, b_gu = time_launches(torch, lambda: hip.hip_swiglu_linear_func(xf5, layer5.gate_proj.weight, layer5.up_proj.weight), n=5, reps=5, warmup=2)
        e_gu = mfma_entry("gemm_tiles_kernel<swiglu> (gate/up projection + SwiGLU), config 5 (32768 x 2 x 8192 x 2048)", 4 * T5 * H5 * I5, m_gu, b_gu, None, sustained)
        h5 = hip.hip_swiglu_linear_func(xf5, layer5.gate_proj.weight, layer5.up_proj.weight)
        m_d, b_d = time_launches(torch, lambda: hip.hip_linear_func(h5, layer5.down_proj.weight), n=5, reps=5, warmup=2)
        e_d = mfma_entry("gemm_tiles_kernel<plain> (down projection), config 5 (32768 x 2048 x 8192)", 2 * T5 * H5 * I5, m_d, b_d, None, sustained)
        wcat5 = torch.cat([wx5, wy5], 0)
        m_r, b_r = time_launches(torch, lambda: hip.hip_linear_func(xf5, wcat5), n=5, reps=5, warmup=2)
        e_r = mfma_entry("gemm_tiles_kernel<plain> (router projection, both halves: 32768 x 1024 x 2048; arithmetic intensity 669 flop/B), config 5",
                         4 * T5 * H5 * r5, m_r, b_r, None, sustained)
        m_lib, _ = time_launches(torch, lambda: torch.matmul(xf5, wcat5.t()), n=5, reps=3, warmup=2)
        e_r["library_gemm_same_flops_ms"] = m_lib
        wcat_gu = torch.cat([layer5.gate_proj.weight, layer5.up_proj.weight], 0)
        m_lib, _ = time_launches(torch, lambda: torch.matmul(xf5, wcat_gu.t()), n=5, reps=3, warmup=2)
        e_gu["library_gemm_same_flops_ms"] = m_lib
        del wcat_gu
        m_lib, _ = time_launches(torch, lambda: torch.matmul(h5, layer5.down_proj.weight.t()), n=5, reps=3, warmup=2)
        e_d["library_gemm_same_flops_ms"] = m_lib
        m_rt, b_rt = time_launches(torch, router_stage_call(torch, _lib, layer5, xf5, False), n=5, reps=5, warmup=2)
        kernels += [e_gu, e_d, e_r]
        out["layer_c5"] = {"workload": "benchmark config 5: full OmniMoE layer forward, 8x4096 tokens, hidden 2048, intermediate 8192, "
                                       "262144 experts (512x512), top-32, eval-mode BatchNorm whose buffers carry the Zipf(1.1) key bias, seed 4",
                           "ms_per_step": per_algo["auto"]["ms_per_step"], "tokens_per_s": per_algo["auto"]["tokens_per_s"],
                           "with_expert_algo_gather": per_algo["gather"], "on_two_streams": {"ms_per_step": m2, "ms_per_step_best": b2},
                           "router_stage_ms": m_rt,
                           "gate_up_TFLOPs": e_gu["achieved"], "down_TFLOPs": e_d["achieved"], "router_projection_TFLOPs": e_r["achieved"],
                           "frac_of_mfma_peak": {"gate_up": e_gu["frac"], "down": e_d["frac"], "router_projection": e_r["frac"]},
                           "checked": f"{sub} tokens against the oracle (router ids, experts over the selected rows, MLP) before timing"}
        del layer5, h5, wcat5, y5l

    if "expert_c5" in sections or "layer_c5" in sections:
        del x5, up5, down5, wx5, wy5, g5, i5

    if "ref_grid" in sections:
        # The reference's own operator benchmarks (bf16, 1024 tokens), its flop conventions, each beside the same operator
        # composed from torch library ops on this GPU (what the reference's harness calls the PyTorch implementation).
        grid = []
        Tg = 1024
        gen = torch.Generator(device=dev).manual_seed(0)
        for r_, k_ in ((64, 16), (64, 32), (128, 16), (128, 32), (256, 16), (256, 32)):        # tests/test_router.py:103-110
            lx = torch.log_softmax(torch.randn(Tg, r_, device=dev, generator=gen), -1).bfloat16()
            ly = torch.log_softmax(torch.randn(Tg, r_, device=dev, generator=gen), -1).bfloat16()
            sc, ix = hip.hip_omni_router_func(lx, ly, r_, k_)
            ws_, wi_ = oracle.router_select(lx[:64].cpu(), ly[:64].cpu(), r_, k_)
            assert torch.equal(ix[:64].cpu(), wi_) and torch.equal(sc[:64].cpu().float(), ws_.float())
            m, b = time_launches(torch, lambda: hip.hip_omni_router_func(lx, ly, r_, k_))
            mt, _ = time_launches(torch, lambda: (lx[:, :, None] + ly[:, None, :]).view(Tg, -1).topk(k_, dim=-1), n=10, reps=3, warmup=2)
            grid.append({"op": "router", "tokens": Tg, "num_keys": r_, "top_k": k_, "ms": m, "ms_best": b, "torch_ops_ms": mt, "speedup": mt / m,
                         "TFLOPs_reference_convention": 4.0 * Tg * r_ * r_ / (m * 1e-3) / 1e12})
        for N_ in (1024, 4096, 16384, 65536):                                                  # tests/test_expert.py:181-187
            k_ = 32
            xg = torch.empty(Tg, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.5, generator=gen)
            ug = torch.empty(N_, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            vg = torch.empty(N_, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            gg = torch.empty(Tg, k_, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            ig = torch.randint(0, N_, (Tg, k_), device=dev, dtype=torch.int32, generator=gen)
            yg = hip.hip_omni_expert_func(xg, ug, vg, gg, ig)
            rows, inv = torch.unique(ig[:64].long(), return_inverse=True)
            wantg = oracle.expert_forward(xg[:64].cpu(), ug[rows].cpu(), vg[rows].cpu(), gg[:64].cpu(), inv.cpu().to(torch.int32))
            torch.testing.assert_close(yg[:64].float().cpu(), wantg.float(), rtol=2e-2, atol=2e-2)
            m, b = time_launches(torch, lambda: hip.hip_omni_expert_func(xg, ug, vg, gg, ig))

            def torch_expert():
                il = ig.long()
                sc_ = torch.einsum("th,tkh->tk", xg, ug[il])
                return torch.einsum("tk,tkh->th", torch.nn.functional.silu(sc_) * gg, vg[il])

            mt, _ = time_launches(torch, torch_expert, n=10, reps=3, warmup=2)
            grid.append({"op": "expert", "tokens": Tg, "hidden": 1024, "num_experts": N_, "top_k": k_, "ms": m, "ms_best": b, "torch_ops_ms": mt, "speedup": mt / m,
                         "TFLOPs_reference_convention": 4.0 * Tg * k_ * 1024 / (m * 1e-3) / 1e12,
                         "algorithmic_GBs": expert_alg_bytes(Tg, 1024, k_) / (m * 1e-3) / 1e9})
            del xg, ug, vg, gg, ig, yg
        gen = torch.Generator(device=dev).manual_seed(42)
        for I_ in (1024, 4096, 16384, 65536):                                                  # tests/test_mlp.py:144-150
            xg = torch.empty(Tg, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.5, generator=gen)
            wg_ = torch.empty(I_, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            wu_ = torch.empty(I_, 1024, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            wd_ = torch.empty(1024, I_, device=dev, dtype=torch.bfloat16).normal_(0, 0.1, generator=gen)
            yg = hip.hip_omni_mlp_func(xg, wg_, wu_, wd_)
            wantg = oracle.mlp_forward(xg[:32].cpu().float(), wg_.cpu().float(), wu_.cpu().float(), wd_.cpu().float())
            scale = max(wantg.abs().max().item(), 1.0)
            torch.testing.assert_close(yg[:32].float().cpu() / scale, wantg / scale, rtol=2e-2, atol=2e-2)
            m, b = time_launches(torch, lambda: hip.hip_omni_mlp_func(xg, wg_, wu_, wd_), n=20)
            mt, _ = time_launches(torch, lambda: torch.matmul(torch.nn.functional.silu(torch.matmul(xg, wg_.t())) * torch.matmul(xg, wu_.t()), wd_.t()), n=10, reps=3, warmup=2)
            grid.append({"op": "mlp", "tokens": Tg, "hidden": 1024, "intermediate": I_, "ms": m, "ms_best": b, "torch_ops_ms": mt, "speedup": mt / m,
                         "TFLOPs_reference_convention": 6.0 * Tg * 1024 * I_ / (m * 1e-3) / 1e12})
            del xg, wg_, wu_, wd_, yg
        out["ref_grid"] = grid

    if kernels:
        out["kernels"] = kernels
        out["traffic_source"] = TRAFFIC_SOURCE

    if "cpu" in sections:
        # the oracle (torch CPU restatement of the reference's PyTorch layer) on the host cores, on the whole workload
        # (all 4096 tokens, train-mode BatchNorm), repeated for ~10 s
        threads = min(16, os.cpu_count() or 1)
        torch.set_num_threads(threads)
        reps, t0 = 0, time.perf_counter()
        while time.perf_counter() - t0 < 10.0 or reps < 2:
            bx, by = oracle.BNState.fresh(layer.num_expert_sqrt), oracle.BNState.fresh(layer.num_expert_sqrt)
            oracle.moe_forward(x, w, bx, by, k, training=True, expert_compute_dtype=None)
            reps += 1
        dt = time.perf_counter() - t0
        out["cpu_baseline"] = {"value": reps * T / dt, "unit": "tokens/s", "cores": torch.get_num_threads(), "kind": "port",
                               "host_logical_cpus": os.cpu_count(), "cpu_model": cpu_model(),
                               "sample": f"{reps} forwards of the whole workload (4096 tokens) in {dt:.1f} s, bf16 torch CPU ops on "
                                         f"{torch.get_num_threads()} threads (oracle restatement of OmniMoE_Torch.forward)"}
    if a.details:
        with open(a.details, "w") as f:
            json.dump(out, f, indent=1)
    print(headline(out))


if __name__ == "__main__":
    main()
