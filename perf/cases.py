"""The work this library is used for, as cases that can be timed and compared.

A case is a dict of plain values.  ``kind`` names the public entry point that it goes through:

  infer    ``OmniMoE.forward`` under ``torch.no_grad()``: serving (eval mode) or a forward with batch statistics (train mode)
  train    ``OmniMoE.forward`` with autograd recording, then ``backward``: one training step's gradients
  experts  ``hip_omni_expert_func``, forward, or forward and backward (``grad``)
  router   ``hip_omni_router_fwd_func``: hidden states to gates and expert ids
  mlp      ``hip_omni_mlp_func``: the shared SwiGLU MLP, without autograd

Sizes: ``tokens`` T, ``hidden`` H, ``inter`` I (intermediate size), ``experts`` N, ``top_k`` k; ``dtype`` is the storage type of
activations and weights.  ``norm`` is the mode of the router's BatchNorm ("batch" statistics as in training, or the "running"
buffers as in serving).  ``skew`` is the Zipf exponent of the keys' popularity (0: every expert is as likely as any other).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "omni-moe_amd"))

from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig  # noqa: E402
from omni_moe.ops.hip import hip_omni_expert_func, hip_omni_mlp_func, hip_omni_router_fwd_func  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}

#: Work of the largest listed case (tokens x hidden x intermediate, and table rows x hidden): no drawn case goes beyond it.
MOST_WORK = 32768 * 2048 * 8192
MOST_TABLE = 262144 * 2048


def listed():
    layer = {"kind": "infer", "hidden": 1024, "inter": 4096, "experts": 4096, "top_k": 16, "dtype": "bf16", "norm": "running", "skew": 0.0}
    step = dict(layer, kind="train", norm="batch")
    return [
        # one sequence generating token by token: launches and the weights' one trip through memory
        dict(layer, name="decode 1", tokens=1),
        # a small batch of sequences decoded together
        dict(layer, name="decode 48", tokens=48),
        # one prompt of ordinary, ragged length, in the other 16-bit type
        dict(layer, name="prefill 613 f16", tokens=613, dtype="f16"),
        # the README's layer: 1 x 4096 tokens with batch statistics, the forward that bench.py reports
        dict(layer, name="forward 4096", tokens=4096, norm="batch"),
        # the large layer: 8 x 4096 tokens, 512 x 512 keys of Zipf-like popularity
        dict(layer, name="prefill 32768 large", tokens=32768, hidden=2048, inter=8192, experts=262144, top_k=32, skew=1.1),
        # the small single-precision layer that is also checked against the CPU path
        dict(layer, name="forward 512 f32", tokens=512, hidden=256, inter=1024, experts=1024, top_k=8, dtype="f32", norm="batch"),
        # a training step of the README's layer
        dict(step, name="train 4096", tokens=4096),
        # a training step of a smaller layer on a ragged micro-batch
        dict(step, name="train 1000 small", tokens=1000, hidden=512, inter=2048, experts=1024, top_k=8),
        # the routed experts alone, for a model that brings its own router and MLP
        {"kind": "experts", "name": "experts 16384", "tokens": 16384, "hidden": 1024, "experts": 4096, "top_k": 16, "dtype": "bf16", "grad": False},
        # ... and trained: few tokens over a large table
        {"kind": "experts", "name": "experts 1024 grad", "tokens": 1024, "hidden": 1024, "experts": 16384, "top_k": 32, "dtype": "bf16", "grad": True},
        # the router alone
        {"kind": "router", "name": "router 4096", "tokens": 4096, "hidden": 1024, "experts": 4096, "top_k": 16, "dtype": "bf16", "norm": "batch"},
        # the MLP alone, few tokens through a wide intermediate
        {"kind": "mlp", "name": "mlp 1024 wide", "tokens": 1024, "hidden": 1024, "inter": 16384, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case: token counts of any value, hidden sizes of the tensor-core kind and (one in eight) merely of whole 16-byte
    rows, key grids from 16 x 16 to 512 x 512 (now and then with experts beyond the square), top-k 2 to 32."""
    kind = rng.choice(["infer"] * 6 + ["train"] * 2 + ["experts"] * 2 + ["router", "mlp"])
    dtype = rng.choice(["bf16"] * 6 + ["f16", "f32"])
    while True:
        hidden = rng.choice([256, 512, 768, 1024, 1024, 1280, 2048]) if rng.random() < 0.875 else 8 * rng.randint(25, 200)
        inter = rng.choice([2, 3, 4, 4]) * hidden
        keys = _log_int(rng, 16, 512)
        experts = keys * keys + (rng.randint(1, 2 * keys) if rng.random() < 0.25 else 0)
        top_k = 2 * _log_int(rng, 1, 16)
        most = {"infer": 32768, "train": 8192, "experts": 32768, "router": 32768, "mlp": 32768}[kind]
        tokens = _log_int(rng, 1 if kind in ("infer", "mlp") else 64, most)
        limit = MOST_WORK // (16 if dtype == "f32" else 1) // (3 if kind == "train" else 1)      # single precision runs at a sixteenth of the matrix rate
        if tokens * hidden * inter <= limit and experts * hidden <= MOST_TABLE // (8 if kind == "train" or dtype == "f32" else 1):
            break
    case = {"kind": kind, "tokens": tokens, "hidden": hidden, "dtype": dtype}
    if kind != "mlp":
        case.update(experts=experts, top_k=top_k)
    if kind in ("infer", "train", "mlp"):
        case.update(inter=inter)
    if kind in ("infer", "router"):
        case.update(norm="batch" if tokens >= 64 and rng.random() < 0.25 else "running")
    if kind == "infer":
        case.update(skew=rng.choice([0.0, 0.0, 1.1]) if case["norm"] == "running" else 0.0)
    if kind == "train":
        case.update(norm="batch", skew=0.0)
    if kind == "experts":
        case.update(grad=rng.random() < 0.5)
    return case


def _normal(gen, dtype, std, *shape):
    return torch.empty(*shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=gen)


def prepare(case, seed):
    """Inputs x ~ N(0,1) and weights ~ N(0, 0.02) as in the layer's configurations; a layer is an ``OmniMoE`` module that lives on."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    kind, T, H = case["kind"], case["tokens"], case["hidden"]
    if kind in ("infer", "train"):
        with torch.device("meta"):
            layer = OmniMoE(OmniMoEConfig(H, case["inter"], "silu", case["experts"], case["top_k"]))
        layer = layer.to(dtype).to_empty(device="cuda")
        with torch.no_grad():
            for p in layer.parameters():
                p.normal_(0.0, 0.02, generator=gen)
        for norm in (layer.router_norm_x, layer.router_norm_y):
            norm.reset_running_stats()
            if case["norm"] == "running":
                # what training has left there: the variance of x W^T, and per key a bias that makes key i chosen like 1 / (1 + i)^skew
                norm.running_var.fill_(H * 0.02 ** 2)
                norm.running_mean.copy_(case["skew"] * 0.02 * H ** 0.5 * torch.log1p(torch.arange(layer.num_expert_sqrt)))
        layer.train(case["norm"] == "batch")
        state = {"kind": kind, "layer": layer, "x": _normal(gen, dtype, 1.0, 1, T, H)}
        if kind == "train":
            state["x"].requires_grad_()
            state["dy"] = _normal(gen, dtype, 1.0, 1, T, H)
        return state
    state = {"kind": kind, "x": _normal(gen, dtype, 1.0, T, H)}
    if kind == "experts":
        N, k = case["experts"], case["top_k"]
        state.update(up=_normal(gen, dtype, 0.02, N, H), down=_normal(gen, dtype, 0.02, N, H),
                     gates=torch.softmax(_normal(gen, torch.float32, 1.0, T, k), -1).to(dtype),
                     ids=torch.randint(0, N, (T, k), device="cuda", dtype=torch.int32, generator=gen))
        if case["grad"]:
            state["dy"] = _normal(gen, dtype, 1.0, T, H)
            for n in ("x", "up", "down", "gates"):
                state[n].requires_grad_()
    elif kind == "router":
        r = math.isqrt(case["experts"])
        state.update(wx=_normal(gen, dtype, H ** -0.5, r, H), wy=_normal(gen, dtype, H ** -0.5, r, H), k=case["top_k"], training=case["norm"] == "batch",
                     stats=[torch.zeros(r, device="cuda", dtype=dtype), torch.ones(r, device="cuda", dtype=dtype), torch.zeros((), device="cuda", dtype=torch.int64),
                            torch.zeros(r, device="cuda", dtype=dtype), torch.ones(r, device="cuda", dtype=dtype), torch.zeros((), device="cuda", dtype=torch.int64)])
    else:
        I = case["inter"]
        state.update(wg=_normal(gen, dtype, 0.02, I, H), wu=_normal(gen, dtype, 0.02, I, H), wd=_normal(gen, dtype, 0.02, H, I))
    return state


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            return {"y": state["layer"](state["x"]), "buffers": list(state["layer"].buffers())}
    if kind == "train":
        layer, x = state["layer"], state["x"]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        y = layer(x)
        y.backward(state["dy"])
        return {"y": y.detach(), "dx": x.grad, "grads": [p.grad for p in layer.parameters()], "buffers": list(layer.buffers())}
    if kind == "experts":
        leaves = [state[n] for n in ("x", "up", "down", "gates")]
        if "dy" not in state:
            with torch.no_grad():
                return hip_omni_expert_func(*leaves, state["ids"])
        for t in leaves:
            t.grad = None
        y = hip_omni_expert_func(*leaves, state["ids"])
        y.backward(state["dy"])
        return {"y": y.detach(), "grads": [t.grad for t in leaves]}
    with torch.no_grad():
        if kind == "router":
            gates, ids = hip_omni_router_fwd_func(state["x"], state["wx"], state["wy"], *state["stats"], state["k"], training=state["training"])
            return {"gates": gates, "ids": ids, "stats": state["stats"]}
        return hip_omni_mlp_func(state["x"], state["wg"], state["wu"], state["wd"])


def work(case):
    """Every operand once: activations, weights, and of the expert tables the rows that are selected (gradients of tables are dense)."""
    T, H, es = case["tokens"], case["hidden"], BYTES[case["dtype"]]
    I, N, k = case.get("inter", 0), case.get("experts", 0), case.get("top_k", 0)
    r = math.isqrt(N)
    kind = case["kind"]
    pairs = T * k
    rows = N * -math.expm1(pairs * math.log1p(-1.0 / N)) if N > 1 else float(N)       # distinct rows of so many uniform choices
    if case.get("skew"):
        rows = min(rows, 8 * r)                                                       # a Zipf(1.1) router keeps to about 8 rows a key
    mlp, router, pair = T * H * I, T * H * r, pairs * H
    if kind == "infer":
        return {"bytes": (2 * T * H + 3 * H * I + 2 * r * H + 2 * rows * H) * es, "flops": 6 * mlp + 4 * router + 4 * pair}
    if kind == "train":
        weights = 3 * H * I + 2 * r * H
        return {"bytes": (4 * T * H + 2 * weights + 2 * rows * H + 2 * N * H) * es, "flops": 18 * mlp + 12 * router + 12 * pair}
    if kind == "experts":
        fwd = (2 * T * H + 2 * rows * H + pairs) * es + 4 * pairs
        return {"bytes": fwd + ((2 * T * H + 2 * N * H + pairs) * es if case["grad"] else 0), "flops": (12 if case["grad"] else 4) * pair}
    if kind == "router":
        return {"bytes": (T * H + 2 * r * H + pairs) * es + 4 * pairs, "flops": 4 * router}
    return {"bytes": (2 * T * H + 3 * H * I) * es, "flops": 6 * mlp}


def tolerance(case):
    """Rounding to the storage type at the points where the operators store (once per operand and per result), sums in 32 bits in
    any order.  A last-bit difference in a router score may also pick the other of two nearly equal experts for a token: of little
    weight in a sum (the least of a token's gates), and in ids a share of a per cent at most."""
    rel = {"bf16": 1e-2, "f16": 2e-3, "f32": 1e-5}[case["dtype"]]
    most = {"bf16": 0.4, "f16": 0.1, "f32": 5e-3}[case["dtype"]]
    if case["kind"] == "train":
        return {"rel": {"bf16": 2e-2, "f16": 1e-2, "f32": 1e-4}[case["dtype"]], "max": 0.99 if case["dtype"] != "f32" else 0.05}
    if case["kind"] == "router":
        return {"rel": rel, "max": 0.99, "differ": 0.01}
    return {"rel": rel, "max": most}
