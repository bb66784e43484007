"""GPU parity of the MLP, the fused router and the whole OmniMoE layer against the CPU oracle."""
import pytest
import torch

from oracle import omni_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _inference():
    """These tests cover the fused forward; with autograd recording the module is one
    differentiable node instead (tests/test_gpu_backward.py)."""
    with torch.no_grad():
        yield


def _ops():
    from omni_moe.ops import hip
    return hip


def _elsewhere(t, device):
    """t's values, contiguous, from one element past a 16-byte boundary on: a parameter that is a view into a flat buffer."""
    flat = torch.empty(t.numel() + 1, device=device, dtype=t.dtype)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    assert out.is_contiguous() and out.data_ptr() % 16 == t.element_size()
    return out


# the first four are the reference's benchmark grid (tests/test_mlp.py:144-150): intermediate 1024 .. 65536
MLP_CASES = [(1024, 1024, 1024), (1024, 1024, 4096), (1024, 1024, 16384), (1024, 1024, 65536), (4096, 1024, 4096), (4100, 1024, 4096),
             (333, 256, 1000), (128, 64, 128), (512, 2048, 8192), (5, 8, 8),
             (8192, 128, 4096), (8200, 192, 2048)]      # streaming gate/up kernel with two and three K tiles per output tile, four tiles per block


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", MLP_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}")
def test_mlp_matches_oracle(case, dtype, device):
    T, H, I = case
    g = torch.Generator().manual_seed(42)
    # reference benchmark distribution (tests/test_mlp.py:72-84): x~N(0,0.5), W~N(0,0.1) -- scaled
    # down for f16 at large I so the sums stay in range
    ws = 0.1 if dtype == torch.bfloat16 or I <= 1024 else 0.03
    x = (torch.randn(T, H, generator=g) * 0.5).to(dtype)
    wg, wu = ((torch.randn(I, H, generator=g) * ws).to(dtype) for _ in range(2))
    wd = (torch.randn(H, I, generator=g) * ws).to(dtype)
    res = torch.randn(T, H, generator=g).to(dtype)
    print(f"mlp T={T} H={H} I={I} {dtype}", flush=True)
    want = oracle.mlp_forward(x.float(), wg.float(), wu.float(), wd.float())      # fp32 everywhere
    d = [t.to(device) for t in (x, wg, wu, wd)]
    got = _ops().hip_omni_mlp_func(*d).cpu().float()
    scale = want.abs().max().item()
    # bf16 storage of gate/up/h contributes ~2^-8 relative noise per term; compare on the output's scale
    assert (got - want).abs().max().item() <= 2e-2 * max(scale, 1.0)
    torch.testing.assert_close(got / max(scale, 1.0), want / max(scale, 1.0), rtol=2e-2, atol=2e-2)
    got_r = _ops().hip_omni_mlp_func(*d, residual=res.to(device)).cpu().float()
    want_r = got.to(dtype).float() + res.float()
    torch.testing.assert_close(got_r, want_r.to(dtype).float(), rtol=1e-2, atol=1e-2 * max(scale, 1.0))


@pytest.mark.parametrize("case", [(512, 256, 1024), (300, 100, 260), (64, 1024, 512)], ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}")
def test_mlp_fp32_matches_oracle(case, device):
    T, H, I = case
    g = torch.Generator().manual_seed(7)
    x = torch.randn(T, H, generator=g)
    wg, wu, wd = torch.randn(I, H, generator=g) * 0.05, torch.randn(I, H, generator=g) * 0.05, torch.randn(H, I, generator=g) * 0.05
    res = torch.randn(T, H, generator=g)
    print(f"mlp fp32 T={T} H={H} I={I}", flush=True)
    want = oracle.mlp_forward(x.double(), wg.double(), wu.double(), wd.double()).float()
    d = [t.to(device) for t in (x, wg, wu, wd)]
    got = _ops().hip_omni_mlp_func(*d).cpu()
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-5 * max(1.0, want.abs().max().item()))
    got_r = _ops().hip_omni_mlp_func(*d, residual=res.to(device)).cpu()
    torch.testing.assert_close(got_r, want + res, rtol=1e-4, atol=1e-5 * max(1.0, want.abs().max().item()))


# the last two make the projection GEMM pick its 128 x 128 and 256 x 256 tiles (statistics epilogue included)
ROUTER_FWD_CASES = [(4096, 1024, 64, 16), (1024, 256, 32, 8), (2048, 2048, 512, 32), (300, 520, 36, 10), (300, 576, 36, 10),
                    (4096, 256, 512, 32), (16384, 256, 512, 32), (200, 128, 1300, 16)]      # last: more than 1024 keys per half


def _bn_buffers(r, dtype, device=None):
    m, v = torch.zeros(r, dtype=dtype), torch.ones(r, dtype=dtype)
    n = torch.zeros((), dtype=torch.long)
    return [t.to(device) if device else t for t in (m, v, n)]


@pytest.mark.parametrize("training", [True, False], ids=["train", "eval"])
@pytest.mark.parametrize("case", ROUTER_FWD_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-r{c[2]}-k{c[3]}")
def test_router_fwd_matches_oracle(case, training, device):
    T, H, r, k = case
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(1)
    x = torch.randn(T, H, generator=g).to(dtype)
    wx, wy = ((torch.randn(r, H, generator=g) / H ** 0.5).to(dtype) for _ in range(2))
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    if not training:   # eval: give the buffers content (a per-key bias and scale)
        for b in (bx, by):
            b.running_mean.copy_(torch.randn(r, generator=g) * 0.3)
            b.running_var.copy_(torch.rand(r, generator=g) + 0.5)
    dbx = [bx.running_mean.clone().to(device), bx.running_var.clone().to(device), torch.zeros((), dtype=torch.long, device=device)]
    dby = [by.running_mean.clone().to(device), by.running_var.clone().to(device), torch.zeros((), dtype=torch.long, device=device)]
    print(f"router_fwd T={T} H={H} r={r} k={k} training={training}", flush=True)
    want_g, want_i, want_s = oracle.router_forward(x, wx, wy, bx, by, k, training)
    got_g, got_i, got_s = _ops().hip_omni_router_fwd_func(x.to(device), wx.to(device), wy.to(device), *dbx, *dby, k,
                                                          training=training, return_scores=True)
    torch.cuda.synchronize()
    got_i, got_g, got_s = got_i.cpu(), got_g.cpu(), got_s.cpu()
    # internal consistency, exact: the gate is exp of the score, scores descend
    assert torch.equal(got_g.float(), torch.exp(got_s.float()).to(dtype).float())
    assert (got_s[:, :-1].float() >= got_s[:, 1:].float()).all()
    # end-to-end index agreement with the oracle (the projections differ in fp32 summation
    # order, so a bf16 rounding can flip): >= 99.9 % of the per-token expert sets
    same_pos = (got_i == want_i).float().mean().item()
    a, b = got_i.sort(-1).values, want_i.sort(-1).values
    set_agree = (a == b).float().mean().item()
    print(f"   position agreement {same_pos:.5f}, set agreement {set_agree:.5f}")
    assert set_agree >= 0.999, set_agree
    assert same_pos >= 0.99, same_pos
    torch.testing.assert_close(got_g.float(), want_g.float(), rtol=2e-2, atol=2e-2)
    # running statistics
    if training:
        torch.testing.assert_close(dbx[0].cpu(), bx.running_mean, rtol=1e-3, atol=1e-4)
        torch.testing.assert_close(dbx[1].cpu(), bx.running_var, rtol=1e-3, atol=1e-4)
        torch.testing.assert_close(dby[1].cpu(), by.running_var, rtol=1e-3, atol=1e-4)
        assert dbx[2].item() == 1 and dby[2].item() == 1
    else:
        assert torch.equal(dbx[0].cpu(), bx.running_mean) and dbx[2].item() == 0


# Statistics merged by the selecting blocks: both block sizes, at the border between them, two candidates to a lane, an odd number of keys, a partial strip
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", [(2048, 256, 64, 32), (2049, 256, 64, 32), (4096, 128, 64, 16), (1029, 256, 33, 8), (70, 256, 64, 2), (2, 128, 16, 4)], ids=lambda c: "T%d-H%d-r%d-k%d" % c)
def test_router_fwd_merges_statistics_where_it_selects(case, dtype, device):
    """Gates and ids against the oracle (a last-bit difference of a score may pick the other of two nearly equal experts: one in a hundred at most), buffers and counts
    after two batches."""
    T, H, r, k = case
    g = torch.Generator().manual_seed(T + r)
    wx, wy = ((torch.randn(r, H, generator=g) / H ** 0.5).to(dtype) for _ in range(2))
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    dbx, dby = _bn_buffers(r, torch.float32, device), _bn_buffers(r, torch.float32, device)
    print(f"router_fwd merged T={T} H={H} r={r} k={k} {dtype}", flush=True)
    for _ in range(2):
        x = torch.randn(T, H, generator=g).to(dtype)
        want_g, want_i, _ = oracle.router_forward(x, wx, wy, bx, by, k, True)
        got_g, got_i = _ops().hip_omni_router_fwd_func(x.to(device), wx.to(device), wy.to(device), *dbx, *dby, k, training=True)
        if T > 2:                                       # (two tokens normalise to +-1: every key ties)
            assert (got_i.cpu().sort(-1).values == want_i.sort(-1).values).float().mean().item() >= 0.99
            torch.testing.assert_close(got_g.cpu().float(), want_g.float(), rtol=2e-2, atol=2e-2)
    for d, b in ((dbx, bx), (dby, by)):
        torch.testing.assert_close(d[0].cpu(), b.running_mean, rtol=1e-3, atol=1e-4)
        torch.testing.assert_close(d[1].cpu(), b.running_var, rtol=1e-3, atol=1e-4)
        assert d[2].item() == 2


def _cancelling_strips(T, H, g):
    """Rows whose first column has half of the whole strips of 32 in pairs of +-values up to 2^59, which cancel exactly, and values of about 1000 in the others: every order of the
    strips' double sums loses other bits of what is left."""
    strips = (T + 31) // 32
    big = torch.zeros(strips)
    order = torch.randperm(T // 32, generator=g)
    for a, b in zip(order[0::4].tolist(), order[1::4].tolist()):        # half of the whole strips in pairs
        big[a] = (1.0 + torch.rand((), generator=g)) * 2.0 ** torch.randint(50, 59, (), generator=g)
        big[b] = -big[a]
    x = torch.randn(T, H, generator=g)
    x[:, 0] = torch.where(big != 0, big, 1000.0 * torch.randn(strips, generator=g)).repeat_interleave(32)[:T]
    return x


# eight waves a block and sixteen, 4 to 64 sums of a column, an odd number of keys, a partial strip, more than 64 strips
@pytest.mark.parametrize("case", [(70, 60), (700, 2), (700, 3), (2100, 6), (700, 12), (700, 20), (2100, 33), (1000, 60), (2100, 60)], ids=lambda c: "T%d-r%d" % c)
def test_batch_statistics_on_one_stream_and_two(case, device):
    """A layer on one stream merges the batch statistics where it selects, on two in a launch of their own: one order of the double sums, so the same buffers to the
    bit also where that order shows."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, r = case
    H, I, k = 128, 256, 2
    print(f"statistics on one stream and two T={T} r={r} k={k}", flush=True)
    g = torch.Generator().manual_seed(T + r)
    x = _cancelling_strips(T, H, g)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", r * r, k)).to(device=device, dtype=torch.bfloat16)
    norms = layer.router_norm_x.float(), layer.router_norm_y.float()
    for w in (layer.router_gate_x.weight, layer.router_gate_y.weight):
        w.copy_(torch.randn(r, H, generator=g) * H ** -0.5)
        w[:, 0] = 1.0
    layer.overlap_min_work = 0
    x = x.to(device=device, dtype=torch.bfloat16)
    left = []
    for two in (False, True):
        layer.overlap_branches = two
        for n in norms:
            n.reset_running_stats()
        layer(x[None])
        left.append([b.clone() for n in norms for b in n.buffers()])
    stats = [b for n in norms for b in (torch.zeros_like(n.running_mean), torch.ones_like(n.running_var), torch.zeros_like(n.num_batches_tracked))]
    _ops().hip_omni_router_fwd_func(x, layer.router_gate_x.weight, layer.router_gate_y.weight, *stats, k, training=True)
    assert all(torch.isfinite(b).all() for b in stats)
    for one, two, alone in zip(*left, stats):
        assert torch.equal(one, two) and torch.equal(one, alone)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", [(300, 128, 16, 8), (2100, 128, 64, 16)], ids=lambda c: "T%d-H%d-r%d-k%d" % c)
def test_router_fwd_cumulative_average_where_it_selects(case, dtype, device):
    """momentum=None with the statistics merged by the selecting blocks: the factor 1 / (batches so far + 1) is read before the count moves on."""
    T, H, r, k = case
    g = torch.Generator().manual_seed(T)
    wx, wy = ((torch.randn(r, H, generator=g) / H ** 0.5).to(dtype) for _ in range(2))
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    dbx, dby = _bn_buffers(r, torch.float32, device), _bn_buffers(r, torch.float32, device)
    print(f"router_fwd cumulative T={T} H={H} r={r} k={k} {dtype}", flush=True)
    for step in range(3):
        x = (torch.randn(T, H, generator=g) * (1.0 + step)).to(dtype)
        oracle.router_forward(x, wx, wy, bx, by, k, True, momentum=None)
        _ops().hip_omni_router_fwd_func(x.to(device), wx.to(device), wy.to(device), *dbx, *dby, k, training=True, momentum=None)
        for d, b in ((dbx, bx), (dby, by)):
            torch.testing.assert_close(d[0].cpu(), b.running_mean, rtol=1e-3, atol=3e-4)       # (three times the spread of the test above in the last batch)
            torch.testing.assert_close(d[1].cpu(), b.running_var, rtol=1e-3, atol=1e-4)
            assert d[2].item() == step + 1


def test_router_fwd_select_is_exact_given_same_logprobs(device):
    """Feeding the oracle's selection the device's own scores must reproduce the device's ids
    bit for bit: run the fused router, rebuild the log-probs it saw from its z, compare."""
    T, H, r, k = 1024, 512, 64, 16
    g = torch.Generator().manual_seed(5)
    x = torch.randn(T, H, generator=g).bfloat16()
    wx, wy = ((torch.randn(r, H, generator=g) / H ** 0.5).bfloat16() for _ in range(2))
    hip = _ops()
    z = hip.hip_linear_func(x.to(device), torch.cat([wx, wy]).to(device)).cpu()       # same GEMM kernel
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    px = oracle.log_softmax(oracle.batch_norm(z[:, :r].contiguous(), bx.running_mean, bx.running_var, True))
    py = oracle.log_softmax(oracle.batch_norm(z[:, r:].contiguous(), by.running_mean, by.running_var, True))
    want_s, want_i = oracle.router_select(px, py, r, k)
    d = _bn_buffers(r, torch.float32, device) + _bn_buffers(r, torch.float32, device)
    _, got_i, got_s = hip.hip_omni_router_fwd_func(x.to(device), wx.to(device), wy.to(device), *d, k, training=True, return_scores=True)
    agree = (got_i.cpu() == want_i).float().mean().item()
    print(f"   agreement given device z: {agree:.6f}")
    assert agree >= 0.9995          # only exp/log ulp differences between host and device libm remain


LAYER_CASES = [
    # (T, H, I, N, k, seed)
    (96, 8192, 256, 64, 4, 5),         # expert rows of 16 KiB: the split kernels in two column blocks
    (512, 256, 1024, 1024, 8, 0),      # benchmark config 1 shape, in bf16
    (4096, 1024, 4096, 4096, 16, 3),   # benchmark config 4 (README shape)
    (300, 128, 256, 1000, 8, 1),       # N not a square: r = floor(sqrt(N)) = 31 (omni_moe.py:38), odd, ids < 961
    (300, 128, 256, 1000, 40, 1),      # and k > r, so k' = r
    (64, 64, 128, 50, 6, 2),           # r = 7
    (200, 64, 128, 1100 * 1100, 8, 4), # r = 1100: more keys per half than the select kernels hold in registers
]


@pytest.mark.parametrize("training", [True, False], ids=["train", "eval"])
@pytest.mark.parametrize("case", LAYER_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_layer_matches_oracle(case, training, device):
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k, seed = case
    x, w = oracle.make_layer_inputs(seed, T, H, I, N)
    r = w.router_gate_x.size(0)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    sd = {"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
          "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
          "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}
    missing, unexpected = layer.load_state_dict(sd, strict=False)
    assert not unexpected and all("router_norm" in m for m in missing)
    layer = layer.to(device=device, dtype=torch.bfloat16)
    layer.train(training)
    print(f"layer T={T} H={H} I={I} N={N} k={k} training={training}", flush=True)
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    want, want_g, want_i = oracle.moe_forward(x, w, bx, by, k, training)
    got = layer(x.to(device))
    torch.cuda.synchronize()
    assert got.shape == x.shape and got.dtype == torch.bfloat16
    got_g, got_i = layer.eval().route(x.view(-1, H).to(device)) if not training else (None, None)
    # tokens whose expert set matches the oracle's must match in value; the others differ by
    # which near-tied expert was picked, which changes y by at most a few gate*|V| -- still small
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2e-2, atol=2e-2)
    # the same bound on the scale of the output (|y| is a few 0.01 at these weights, where a flat 2e-2 says little)
    scale = want.float().abs().max().item()
    assert (got.cpu().float() - want.float()).abs().max().item() <= 2e-2 * scale, scale
    if training:
        assert layer.router_norm_x.num_batches_tracked.item() == 1
        torch.testing.assert_close(layer.router_norm_x.running_mean.float().cpu(), bx.running_mean, rtol=2e-2, atol=2e-3)
    else:
        set_agree = (got_i.cpu().sort(-1).values == want_i.sort(-1).values).float().mean().item()
        print(f"   expert-set agreement {set_agree:.5f}")
        assert set_agree >= 0.999


@pytest.mark.parametrize("training", [True, False], ids=["train", "eval"])
def test_layer_config1_fp32(training, device):
    """benchmark config 1, the reference's CPU-runnable case, at full size in fp32:
    1 x 512 tokens, hidden 256, intermediate 1024, 1024 experts (32 x 32), top-8, seed 0."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = 512, 256, 1024, 1024, 8
    x, w = oracle.make_layer_inputs(0, T, H, I, N, dtype=torch.float32)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    layer.load_state_dict({"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
                           "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
                           "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}, strict=False)
    layer = layer.to(device).train(training)
    bx, by = oracle.BNState.fresh(32), oracle.BNState.fresh(32)
    print(f"layer config 1 fp32 training={training}", flush=True)
    want, want_g, want_i = oracle.moe_forward(x, w, bx, by, k, training)
    got = layer(x.to(device))
    torch.cuda.synchronize()
    assert got.dtype == torch.float32
    layer.eval()
    if training:   # route again with the updated buffers on both sides
        want_g, want_i, _ = oracle.router_forward(x.view(-1, H), w.router_gate_x, w.router_gate_y, bx, by, k, False)
    got_g, got_i = layer.route(x.view(-1, H).to(device))
    # fp32 scores: ties practically never occur, so the ids are forced up to fp32 summation order
    set_agree = (got_i.cpu().sort(-1).values == want_i.sort(-1).values).all(-1).float().mean().item()
    print(f"   tokens with identical expert sets: {set_agree:.5f}")
    assert set_agree >= 0.999
    torch.testing.assert_close(got_g.cpu(), want_g, rtol=1e-3, atol=1e-6)
    same = (got_i.cpu().sort(-1).values == want_i.sort(-1).values).all(-1) if not training else torch.ones(T, dtype=torch.bool)
    torch.testing.assert_close(got.cpu().view(-1, H)[same], want.view(-1, H)[same], rtol=1e-3, atol=2e-5)
    if training:
        torch.testing.assert_close(layer.router_norm_x.running_mean.cpu(), bx.running_mean, rtol=1e-4, atol=1e-6)
        torch.testing.assert_close(layer.router_norm_y.running_var.cpu(), by.running_var, rtol=1e-4, atol=1e-6)


def test_layer_config5_large_skewed(device):
    """benchmark config 5: 8 x 4096 tokens, hidden 2048, intermediate 8192, 262144 experts
    (512 x 512 keys), top-32, bf16, router key popularity ~ Zipf(1.1), seed 4.

    The reference's router has no bias (omni_moe.py:47-52), so the per-key bias b_i = -1.1*ln(1+i)
    enters through eval-mode BatchNorm buffers: running_mean = -b, running_var = 1 - eps.  The whole
    batch runs on the GPU; the oracle checks a token subset (eval mode is token-independent) and the
    schedule of all 1M pairs."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k, r = 32768, 2048, 8192, 262144, 32, 512
    g = torch.Generator().manual_seed(4)
    n = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16()
    x = n(8, 4096, H)
    w = oracle.MoEWeights(gate_proj=n(I, H, std=0.02), up_proj=n(I, H, std=0.02), down_proj=n(H, I, std=0.02),
                          router_gate_x=n(r, H, std=0.02), router_gate_y=n(r, H, std=0.02),
                          up_embed=n(N, H, std=0.02), down_embed=n(N, H, std=0.02))
    bias = -1.1 * torch.log1p(torch.arange(r, dtype=torch.float32))
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    layer.load_state_dict({"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
                           "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
                           "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}, strict=False)
    for bn in (layer.router_norm_x, layer.router_norm_y):
        bn.running_mean.copy_(-bias)
        bn.running_var.fill_(1.0 - bn.eps)
    layer = layer.to(device=device, dtype=torch.bfloat16).eval()
    print("layer config 5: 32768 tokens, 262144 experts, top-32", flush=True)
    y = layer(x.to(device))
    gates, ids = layer.route(x.view(-1, H).to(device))
    torch.cuda.synchronize()
    assert y.shape == x.shape and torch.isfinite(y.float()).all()
    # at this size the module keeps to one stream (the GEMMs then take their streaming form); the two-stream schedule, with
    # the other GEMM kernels and the add as a kernel of its own, must give the same bits
    layer.overlap_max_work = 2 ** 62
    assert torch.equal(layer(x.to(device)), y)
    del layer.overlap_max_work
    # schedule of the real, skewed assignment: offsets exact, pairs a grouped permutation
    sched = _ops().hip_omni_schedule_func(ids, N)
    ids_c = ids.cpu()
    want_off, want_pairs, _ = oracle.schedule(ids_c, N)
    assert torch.equal(sched.offsets.cpu(), want_off)
    assert torch.equal(sched.sorted_pair_ids.cpu(), want_pairs)
    seg = (want_off[1:] - want_off[:-1]).float()
    print(f"   pairs per expert: max {int(seg.max())}, mean over used {seg[seg > 0].mean():.1f}, used experts {int((seg > 0).sum())}")
    assert seg.max() > 100 * seg[seg > 0].mean()          # the skew is there
    # oracle on a token subset (buffers as the bf16 module holds them)
    sub = torch.arange(0, T, 128)
    bx = oracle.BNState(layer.router_norm_x.running_mean.float().cpu(), layer.router_norm_x.running_var.float().cpu(), torch.zeros((), dtype=torch.long))
    by = oracle.BNState(layer.router_norm_y.running_mean.float().cpu(), layer.router_norm_y.running_var.float().cpu(), torch.zeros((), dtype=torch.long))
    xs = x.view(-1, H)[sub].unsqueeze(0)
    want, want_g, want_i = oracle.moe_forward(xs, w, bx, by, k, training=False)
    got_i = ids_c[sub]
    set_agree = (got_i.sort(-1).values == want_i.sort(-1).values).float().mean().item()
    print(f"   expert-set agreement on {len(sub)} tokens: {set_agree:.5f}")
    assert set_agree >= 0.999
    torch.testing.assert_close(y.view(-1, H)[sub.to(device)].float().cpu(), want.view(-1, H).float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(gates.cpu()[sub].float(), want_g.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("training", [False, True], ids=["eval", "train"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("two_streams", [False, True], ids=["one-stream", "two-streams"])
def test_layer_expert_term_visible_auto_split(two_streams, dtype, training, device):
    """A layer whose expert branch is as large as its MLP branch (weights ~ N(0, 0.1)) and whose shape makes the layer call
    pick the hidden-split expert algorithm (4096 tokens x 32 = 131072 pairs, tables that overflow one L2): y - mlp must equal
    the oracle's expert term on the expert term's own scale, on one stream and on two.  A layer that dropped or mis-wired
    router -> experts (wrong gates or ids buffer, workspace overlap, missing join) fails here.  In training mode the router
    normalises with the statistics of the whole 4096-token batch, on the device and in the oracle."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = 4096, 512, 512, (1024 if dtype == torch.float32 else 4096), 32
    x, w = oracle.make_layer_inputs(21, T, H, I, N, dtype=dtype, w_std=0.1)
    # the shared MLP scaled down to the size of the expert term (batch statistics flatten the gates: smaller still in training)
    w.down_proj = (w.down_proj.float() * (0.006 if training else 0.03)).to(dtype)
    r = w.router_gate_x.size(0)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    layer.load_state_dict({"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
                           "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
                           "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}, strict=False)
    layer = layer.to(device=device, dtype=dtype).train(training)
    layer.overlap_branches = two_streams
    layer.overlap_min_work = 0
    from omni_moe.ops.hip import _lib
    lib = _lib.load()
    es = 4 if dtype == torch.float32 else 2
    assert lib.omni_expert_workspace_bytes(T, H, N, k, _lib.DTYPE_CODE[dtype], _lib.ALGO_AUTO) == 8 * T * k * 4, "AUTO should pick the split algorithm here"
    print(f"layer with visible expert term, {dtype}, two_streams={two_streams}, training={training}", flush=True)
    xd = x.to(device)
    y = layer(xd).view(-1, H)
    mlp = _ops().hip_omni_mlp_func(xd.view(-1, H), layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight)
    gates, ids = layer.route(xd.view(-1, H))               # training: the same batch again, so the same statistics and ids
    torch.cuda.synchronize()
    bx, by = oracle.BNState.fresh(r), oracle.BNState.fresh(r)
    want_y, want_g, want_i = oracle.moe_forward(x, w, bx, by, k, training=training)
    if training:
        assert layer.router_norm_x.num_batches_tracked.item() == 2
    # the oracle's expert term for the ids the device chose (near-tied scores may resolve differently in bf16)
    want_e = oracle.expert_forward(x.view(-1, H), w.up_embed, w.down_embed, gates.cpu(), ids.cpu()).float()
    e_scale, m_scale = want_e.abs().max().item(), mlp.float().abs().max().item()
    print(f"   max |experts| {e_scale:.3f}, max |mlp| {m_scale:.3f}")
    assert e_scale > 0.15 * m_scale                            # the expert term is visible (batch statistics spread the gates a little thinner)
    got_e = (y.float() - mlp.float()).cpu()
    tol = 1e-4 if dtype == torch.float32 else 2e-2            # bf16: y and mlp are rounded to bf16 on the scale of their sum
    assert (got_e - want_e).abs().max().item() <= tol * (e_scale + m_scale), (got_e - want_e).abs().max().item()
    assert (got_e - want_e).abs().mean().item() <= 0.1 * tol * (e_scale + m_scale)
    same = (ids.cpu().sort(-1).values == want_i.sort(-1).values).all(-1)
    assert same.float().mean().item() >= (0.999 if dtype == torch.float32 else 0.97)
    torch.testing.assert_close(y.cpu().float()[same], want_y.view(-1, H).float()[same], rtol=tol, atol=tol * (e_scale + m_scale))


def _waits_for_side_stream(layer, x):
    """Whether the call forks to the layer's side stream and joins it: what stands on that stream beforehand must then end before the call's work does."""
    layer(x)                                                 # whatever a first call allocates and loads
    side = layer._branch_resources(x.device)[0]
    torch.cuda.synchronize()
    before, after = torch.cuda.Event(), torch.cuda.Event()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)                        # (far longer than the call and its host work)
        before.record()
    layer(x)
    after.record()
    after.synchronize()
    waited = before.query()
    torch.cuda.synchronize()
    return waited


# T, H, I.  16 bits: up to 2^33 token x hidden x intermediate the calls are joint launches on one stream whatever the switches say; beyond it, and in
# single precision and for operands off a 16-byte boundary at any size, they are the two schedules that the switches choose between.
STREAM_CASES = [(torch.bfloat16, (300, 256, 512), True, False), (torch.bfloat16, (300, 256, 512), False, True), (torch.float32, (300, 256, 512), True, True),
                (torch.bfloat16, (2100, 1024, 4096), True, True), (torch.float16, (2100, 1024, 4096), True, True)]


@pytest.mark.parametrize("algo", ["gather", "split"])
@pytest.mark.parametrize("case", STREAM_CASES, ids=lambda c: f"{str(c[0])[6:]}-T{c[1][0]}-H{c[1][1]}-I{c[1][2]}-{'aligned' if c[2] else 'off-boundary'}")
def test_layer_two_streams_equals_one_stream(case, algo, device):
    """The two-stream schedule (router+experts beside the MLP, joined by omni_add_inplace) and the
    one-stream schedule (add fused into the down projection) give bit-identical output, call after call."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    dtype, (T, H, I), aligned, forks = case
    torch.manual_seed(0)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", 1024, 8)).to(device=device, dtype=dtype).eval()
    layer.expert_algo = algo
    layer.overlap_min_work = 0                    # two streams at any size that has them
    x = torch.randn(3, T // 3, H, device=device).to(dtype)
    if not aligned:
        x = _elsewhere(x, device)
    layer.overlap_branches = False
    ref = layer(x)
    assert not _waits_for_side_stream(layer, x)
    layer.overlap_branches = True
    for _ in range(5):
        assert torch.equal(layer(x), ref)
    assert _waits_for_side_stream(layer, x) == (forks or algo == "split")           # (the split algorithm has no joint launches)
    # and next to other work on the caller's stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        z = x * 2
        out = layer(z)
    s.synchronize()
    layer.overlap_branches = False
    assert torch.equal(out, layer(x * 2))


# T, H, I, N, k in single precision: sizes of the joint launches at which the experts alone would be split, or would share a token's slots between four or two waves
F32_STREAM_CASES = [(1100, 256, 1024, 4096, 32), (512, 512, 1024, 4096, 32), (300, 256, 512, 1024, 32), (1000, 512, 1024, 1024, 16)]


@pytest.mark.parametrize("training", [False, True], ids=["eval", "train"])
@pytest.mark.parametrize("aligned", [True, False], ids=["aligned", "off-boundary"])
@pytest.mark.parametrize("algo", ["auto", "gather"])
@pytest.mark.parametrize("case", F32_STREAM_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_layer_fp32_two_streams_equals_one_stream(case, algo, aligned, training, device):
    """In single precision a small layer has joint launches on one stream and the two schedules on two: the experts' sums must run in one order on either, so the
    output is the same to the bit."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = case
    print(f"fp32 streams {case} {algo} aligned={aligned} training={training}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device).train(training)
    g = torch.Generator(device=device).manual_seed(T)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, H ** -0.5, generator=g)
        x = torch.randn(1, T, H, device=device, generator=g)
        if not aligned:
            x = _elsewhere(x, device)
        layer.expert_algo = algo
        layer.overlap_min_work = 0
        layer.overlap_branches = False
        ref = layer(x)
        layer.overlap_branches = True
        assert _waits_for_side_stream(layer, x)
        assert torch.equal(layer(x), ref)


@pytest.mark.parametrize("case", [(70, 64), (512, 32), (700, 64), (1100, 32), (700, 96), (700, 128)], ids=lambda c: "T%d-r%d" % c)
def test_fp32_batch_statistics_on_one_stream_and_two(case, device):
    """The joint launches' blocks merge the batch statistics of a small single-precision layer, on two streams a launch of its own: one order of the double sums."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, r = case
    H, I, k = 128, 256, 8
    print(f"fp32 statistics on one stream and two T={T} r={r}", flush=True)
    g = torch.Generator().manual_seed(T + r)
    x = _cancelling_strips(T, H, g).to(device)[None]
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", r * r, k)).to(device=device)
    norms = layer.router_norm_x, layer.router_norm_y
    for w in (layer.router_gate_x.weight, layer.router_gate_y.weight):
        w.copy_(torch.randn(r, H, generator=g) * H ** -0.5)
        w[:, 0] = 1.0
    layer.overlap_min_work = 0
    left = []
    for two in (False, True):
        layer.overlap_branches = two
        for n in norms:
            n.reset_running_stats()
        layer(x)
        left.append([b.clone() for n in norms for b in n.buffers()])
    assert all(torch.isfinite(b).all() for b in left[0])
    for one, two in zip(*left):
        assert torch.equal(one, two)


def test_layer_copies_and_saves_like_a_plain_module(device, tmp_path):
    """After a two-stream forward (side stream and events in use) a layer is still a plain nn.Module:
    copy.deepcopy, torch.save / torch.load and a state_dict round trip give layers with identical output."""
    import copy
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    torch.manual_seed(3)
    cfg = OmniMoEConfig(1024, 4096, "silu", 1024, 8)
    layer = OmniMoE(cfg).to(device=device, dtype=torch.bfloat16).eval()
    x = torch.randn(2, 1100, 1024, device=device).bfloat16()             # beyond the joint launches: two streams
    assert _waits_for_side_stream(layer, x)
    want = layer(x)
    twin = copy.deepcopy(layer)
    assert torch.equal(twin(x), want)
    path = str(tmp_path / "layer.pt")
    torch.save(layer, path)
    loaded = torch.load(path, weights_only=False)           # a file this test wrote itself
    assert torch.equal(loaded(x), want)
    fresh = OmniMoE(cfg).to(device=device, dtype=torch.bfloat16).eval()
    fresh.load_state_dict(layer.state_dict())
    assert torch.equal(fresh(x), want)
    assert not any(isinstance(v, (torch.cuda.Stream, torch.cuda.Event)) for v in vars(layer).values())


def test_layer_takes_noncontiguous_weights(device):
    """The reference's operators make every tensor argument contiguous (utils.py:47-65); the fused layer call does too."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    torch.manual_seed(4)
    layer = OmniMoE(OmniMoEConfig(128, 256, "silu", 256, 8)).to(device=device, dtype=torch.bfloat16).eval()
    x = torch.randn(1, 300, 128, device=device).bfloat16()
    want = layer(x)
    w = layer.down_proj.weight.data
    layer.down_proj.weight.data = w.t().contiguous().t()    # same values, column-major storage
    assert not layer.down_proj.weight.is_contiguous()
    assert torch.equal(layer(x), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_layer_without_the_native_host_path(dtype, device, monkeypatch):
    """The Python path behind the native one reaches the same kernels: equal bits in both norm modes, and gradients for every parameter."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    from omni_moe.ops.hip import _lib
    torch.manual_seed(6)
    layer = OmniMoE(OmniMoEConfig(128, 256, "silu", 256, 8)).to(device=device, dtype=dtype)
    fresh = {n: b.clone() for n, b in layer.named_buffers()}
    x = torch.randn(1, 300, 128, device=device).to(dtype)

    def both_modes():
        for n, b in layer.named_buffers():
            b.copy_(fresh[n])
        return [layer.train(mode)(x) for mode in (True, False)]

    want = both_modes()
    monkeypatch.setattr(_lib, "_native", _lib.WithoutNative())
    assert all(torch.equal(a, b) for a, b in zip(want, both_modes()))
    with torch.enable_grad():
        layer(x).float().square().sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in layer.parameters())


def test_add_inplace(device):
    hip = _ops()
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        a, b = torch.randn(37, 64, device=device).to(dtype), torch.randn(37, 64, device=device).to(dtype)
        want = (a.float() + b.float()).to(dtype)
        assert torch.equal(hip.hip_add_inplace_func(a.clone(), b), want)
    with pytest.raises(ValueError):
        hip.hip_add_inplace_func(torch.zeros(4, 8, device=device), torch.zeros(4, 9, device=device))


# (M, N, K): the first five select the 128 x 128 output tiles (too few 256 x 256 tiles to fill the chip), ragged M
# included; then a big-tile case, N % 8 == 4 (rows written 8 bytes per lane instead of 16), a ragged last column tile
LINEAR_CASES = [(3300, 1024, 512), (3300, 1024, 640), (3300, 1024, 576), (4096, 1024, 4096), (2049, 1536, 1024),
                (4096, 4096, 256), (300, 100, 264), (333, 1000, 256), (70, 4, 8),
                (300, 62, 128), (129, 1001, 64), (70, 6, 16), (5, 1, 8),       # N % 4 != 0: element-wise stores
                # few 64 x 64 tiles and K >= 512: the K tiles of a block dealt out over its waves (even and ragged shares, tails)
                (4096, 128, 1024), (1000, 104, 512), (130, 72, 640), (64, 64, 4096), (200, 6, 576), (33, 250, 832),
                # the streaming form with a ragged last row tile and with tile counts that are no whole rounds of 256
                (4100, 4096, 512), (3328, 4096, 512), (4353, 4096, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", LINEAR_CASES, ids=lambda c: f"M{c[0]}-N{c[1]}-K{c[2]}")
def test_linear_matches_matmul(case, dtype, device):
    """y = x W^T (+ residual) against an fp64 matmul, over the tile shapes and both store widths."""
    M, N, K = case
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * 0.05).to(dtype)
    res = torch.randn(M, N, generator=g).to(dtype)
    print(f"linear M={M} N={N} K={K} {dtype}", flush=True)
    want = x.double() @ w.double().t()
    got = _ops().hip_linear_func(x.to(device), w.to(device)).cpu()
    # one rounding of an fp32 sum: half an ulp of the storage dtype plus fp32 summation noise
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (got.double() - want).abs()
    assert (err <= ulp * want.abs() * 1.01 + 1e-4 * want.abs().max()).all()
    got_r = _ops().hip_linear_func(x.to(device), w.to(device), residual=res.to(device)).cpu()
    assert torch.equal(got_r, (got.float() + res.float()).to(dtype))


# few 64 x 64 tiles and long K, more of them than CUs, 128 x 128 and 256 x 256 tiles, each with K in whole tiles of 64
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("case", [(130, 72, 640), (1100, 1024, 128), (3300, 1024, 512), (4100, 4096, 128)], ids=lambda c: f"M{c[0]}-N{c[1]}-K{c[2]}")
def test_linear_takes_operands_at_any_address(case, dtype, device):
    """Each operand in turn, and all of them, one element past a 16-byte boundary: one rounding of an fp32 sum, as test_linear_matches_matmul states it,
    and with a residual a second one."""
    M, N, K = case
    g = torch.Generator(device=device).manual_seed(M + K)
    x = torch.randn(M, K, device=device, generator=g).to(dtype)
    w = (torch.randn(N, K, device=device, generator=g) * 0.05).to(dtype)
    res = torch.randn(M, N, device=device, generator=g).to(dtype)
    print(f"linear off the boundary M={M} N={N} K={K} {dtype}", flush=True)
    want = x.double() @ w.double().t()
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    noise = 1e-4 if dtype != torch.float32 else 8 * 2.0 ** -24 * K ** 0.5
    for which in ((0,), (1,), (2,), (0, 1, 2)):
        xo, wo, ro = (_elsewhere(t, device) if i in which else t for i, t in enumerate((x, w, res)))
        got = _ops().hip_linear_func(xo, wo)
        assert ((got.double() - want).abs() <= ulp * want.abs() * 1.01 + noise * want.abs().max()).all(), which
        both = _ops().hip_linear_func(xo, wo, residual=ro).double() - (want + res.double())
        assert (both.abs() <= ulp * (want.abs() + (want + res.double()).abs()) * 1.01 + noise * want.abs().max()).all(), which


# (M, columns per weight matrix, K): streaming kernel (second matrix = whole tiles), K tiles dealt out over the waves, ring kernel, staged kernel
LINEAR2_CASES = [(8192, 512, 256), (16384, 256, 128), (1000, 52, 512), (3000, 200, 192), (300, 36, 40)]


@pytest.mark.parametrize("case", LINEAR2_CASES, ids=lambda c: f"M{c[0]}-N2x{c[1]}-K{c[2]}")
def test_linear_two_weight_matrices_equals_one(case, device):
    """omni_linear2_fwd (the router projection's form: the upper half of the output columns comes from a second weight
    matrix) gives bit for bit what omni_linear_fwd gives on the concatenated weights."""
    from omni_moe.ops.hip import _lib
    M, n, K = case
    g = torch.Generator().manual_seed(M + n)
    x = torch.randn(M, K, generator=g).bfloat16().to(device)
    w_lo = (torch.randn(n, K, generator=g) * 0.05).bfloat16().to(device)
    w_hi = (torch.randn(n, K, generator=g) * 0.05).bfloat16().to(device)
    print(f"linear2 M={M} N=2x{n} K={K}", flush=True)
    want = _ops().hip_linear_func(x, torch.cat([w_lo, w_hi], 0))
    ref = (x.double() @ torch.cat([w_lo, w_hi], 0).double().t())
    assert ((want.double() - ref).abs() <= 2.0 ** -8 * ref.abs() * 1.01 + 1e-4 * ref.abs().max()).all()
    got = torch.empty(M, 2 * n, dtype=torch.bfloat16, device=device)
    lib = _lib.load()
    _lib.check(lib.omni_linear2_fwd(x.data_ptr(), w_lo.data_ptr(), w_hi.data_ptr(), got.data_ptr(), M, K, n,
                                    _lib.DTYPE_CODE[torch.bfloat16], _lib.stream_ptr()), "omni_linear2_fwd")
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("shape", [(150, 256, 512), (1100, 1024, 4096)], ids=["joint", "schedules"])
@pytest.mark.parametrize("overlap", [True, False], ids=["two-streams", "one-stream"])
def test_layer_is_graph_capturable(overlap, shape, device):
    """The library only launches kernels and records/waits events, so a whole layer forward (fork and join
    included) can be captured into a HIP graph; every replay, with eager work in between, equals the eager result.
    The smaller shape is joint launches on one stream whatever the switches say."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    torch.manual_seed(1)
    T, H, I = shape
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", 1024, 8)).to(device=device, dtype=torch.bfloat16).eval()
    layer.overlap_branches = overlap
    layer.overlap_min_work = 0
    x = torch.randn(2, T, H, device=device).bfloat16()
    assert _waits_for_side_stream(layer, x) == (overlap and T > 150)
    want = layer(x).clone()
    warm = torch.cuda.Stream()
    warm.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(warm):
        layer(x)
    torch.cuda.current_stream().wait_stream(warm)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = layer(x)
    for _ in range(4):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(layer(x * 0.5), layer(x * 0.5))      # eager work between the replays
        torch.cuda.synchronize()


def test_layer_cumulative_batch_norm(device):
    """router_norm_x/y with momentum=None (cumulative moving average, factor 1 / num_batches_tracked): three training
    steps on different batches leave the buffers the oracle predicts, counters included."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = 300, 128, 256, 256, 8
    _, w = oracle.make_layer_inputs(9, T, H, I, N, dtype=torch.float32)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
    layer.router_norm_x.momentum = layer.router_norm_y.momentum = None
    layer.load_state_dict({"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
                           "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
                           "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}, strict=False)
    layer = layer.to(device).train()
    bx, by = oracle.BNState.fresh(16), oracle.BNState.fresh(16)
    g = torch.Generator().manual_seed(10)
    for step in range(3):
        x = torch.randn(1, T, H, generator=g) * (1.0 + step)
        want, _, _ = oracle.moe_forward(x, w, bx, by, k, training=True, momentum=None)
        got = layer(x.to(device))
        assert layer.router_norm_x.num_batches_tracked.item() == step + 1 == int(bx.num_batches_tracked)
        torch.testing.assert_close(layer.router_norm_x.running_mean.cpu(), bx.running_mean, rtol=1e-4, atol=1e-6)
        torch.testing.assert_close(layer.router_norm_y.running_var.cpu(), by.running_var, rtol=1e-4, atol=1e-6)
        torch.testing.assert_close(got.cpu(), want, rtol=1e-3, atol=1e-4)
    layer.router_norm_y.momentum = 0.1
    with pytest.raises(ValueError):                               # one momentum for both halves
        layer(x.to(device))


@pytest.mark.parametrize("aligned", [True, False], ids=["joint", "schedules"])
@pytest.mark.parametrize("training", [True, False], ids=["train", "eval"])
@pytest.mark.parametrize("T", [1, 2, 3, 5, 31, 33, 65])
def test_layer_tiny_token_counts(T, training, aligned, device):
    """A handful of tokens (one wave, one partial strip, a single BatchNorm sample in training), on one and on two
    streams: same tolerance as the big cases, and both schedules bit-identical.  Aligned input of these sizes is joint launches either way;
    input off a 16-byte boundary takes the two schedules."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    H, I, N, k = 128, 256, 256, 8
    x, w = oracle.make_layer_inputs(T, T, H, I, N)
    sd = {"gate_proj.weight": w.gate_proj, "up_proj.weight": w.up_proj, "down_proj.weight": w.down_proj,
          "router_gate_x.weight": w.router_gate_x, "router_gate_y.weight": w.router_gate_y,
          "up_embed.weight": w.up_embed, "down_embed.weight": w.down_embed}
    if T == 1 and training:
        # batch statistics of a single sample: nn.BatchNorm1d raises (reference omni_moe.py:70-71), and so do the oracle and the layer
        with pytest.raises(ValueError):
            oracle.moe_forward(x, w, oracle.BNState.fresh(16), oracle.BNState.fresh(16), k, training)
        for overlap in (True, False):
            layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
            layer.load_state_dict(sd, strict=False)
            layer = layer.to(device=device, dtype=torch.bfloat16).train()
            layer.overlap_branches = overlap
            layer.overlap_min_work = 0
            with pytest.raises(ValueError, match="more than 1 value per channel"):
                layer(x.to(device))
            assert layer.router_norm_x.num_batches_tracked.item() == 0
        return
    want, _, _ = oracle.moe_forward(x, w, oracle.BNState.fresh(16), oracle.BNState.fresh(16), k, training)
    outs = []
    for overlap in (True, False):
        layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k))
        layer.load_state_dict(sd, strict=False)
        layer = layer.to(device=device, dtype=torch.bfloat16).train(training)
        layer.overlap_branches = overlap
        layer.overlap_min_work = 0
        xd = x.to(device) if aligned else _elsewhere(x, device)
        outs.append(layer(xd))
        if not training:
            assert _waits_for_side_stream(layer, xd) == (overlap and not aligned)
    torch.testing.assert_close(outs[0].cpu().float(), want.float(), rtol=2e-2, atol=2e-2)
    assert torch.equal(outs[0], outs[1])


# T, H, I, N, k: tiles of 16 rows and their remainders; hidden and intermediate sizes that end inside a block's 64 of K or 16 columns, or
# split K eight ways; 1 to 8 keys per lane, an odd key count, more than 64 candidates, ids beyond the square never chosen
FEW_TOKEN_CASES = [(1, 1024, 4096, 4096, 16), (16, 200, 312, 1000, 8), (17, 1032, 2056, 700, 32), (33, 256, 1024, 90000, 18), (48, 2048, 1024, 17000, 4),
                   (49, 4096, 512, 260, 2), (63, 584, 8, 289, 6), (64, 8, 4096, 300000, 32),
                   # more than 256 blocks in the first launch (one K unit in LDS at a time) and just not, in the second (splits of one unit a wave or of several)
                   (33, 1024, 4104, 4096, 16), (48, 1032, 4032, 256, 8), (48, 1032, 4048, 256, 8), (64, 2048, 8200, 1000, 4)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", FEW_TOKEN_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_few_tokens_match_the_operators(case, dtype, device):
    """At most 64 tokens in eval mode: the joint launches against the router, expert and MLP operators one by one (64-bit MLP), on
    finite data with a non-finite table row that nobody selects.  Tolerance: one rounding of the storage type per stored value (h, the
    MLP's and the experts' sums, the total), on the output's scale."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = case
    print(f"few tokens {case} {dtype}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device, dtype=dtype).eval()
    g = torch.Generator(device=device).manual_seed(T)
    for p in layer.parameters():
        p.normal_(0.0, H ** -0.5, generator=g)
    layer.down_proj.weight.normal_(0.0, I ** -0.5, generator=g)
    for norm in (layer.router_norm_x, layer.router_norm_y):
        norm.running_mean.normal_(0.0, 0.3, generator=g)
        norm.running_var.uniform_(0.5, 2.0, generator=g)
    x = torch.randn(1, T, H, device=device, generator=g).to(dtype)
    gates, ids = layer.route(x[0])
    unused = torch.ones(N, dtype=torch.bool, device=device)
    unused[ids.long().flatten()] = False
    if unused.any():
        row = int(unused.nonzero()[0])
        layer.up_embed.weight[row] = float("nan")
        layer.down_embed.weight[row] = float("inf")
    got = layer(x)[0]
    ops = _ops()
    experts = ops.hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, gates, ids).double()
    xd, wg, wu, wd = (t.double() for t in (x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight))
    h = (torch.nn.functional.silu((xd @ wg.t()).to(dtype).double()) * (xd @ wu.t()).to(dtype).double()).to(dtype).double()
    mlp = h @ wd.t()
    eps = torch.finfo(dtype).eps
    scale = max(1.0, float((mlp + experts).abs().max()))
    assert (got.double() - (mlp + experts)).abs().max().item() <= 4 * eps * scale
    # the MLP operator takes the same launches, with and without a residual
    alone = ops.hip_omni_mlp_func(x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight)
    assert (alone.double() - mlp).abs().max().item() <= 4 * eps * scale
    both = ops.hip_omni_mlp_func(x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight, residual=x[0])
    assert torch.equal(both, (alone.float() + x[0].float()).to(dtype))
    # ids and gates are those of the router operator: the expert term alone (a zero down projection)
    layer.down_proj.weight.zero_()
    assert (layer(x)[0].double() - experts).abs().max().item() <= 4 * eps * max(1.0, float(experts.abs().max()))


# T, H, I, N, k: whole lines of the weights: eight tokens (a half tile of activations) and nine, 16 and 32 and one more; waves without a unit of K (hidden below 512,
# intermediate below 512), a second column tile of the down projection with 8 columns or none (hidden 520, 528), one and two units of K at a time in either launch
FEW_TOKEN_LINES = [(8, 1024, 4096, 4096, 16), (9, 528, 4104, 1000, 8), (7, 520, 72, 64, 2), (24, 264, 264, 1024, 8), (32, 1032, 4104, 4096, 16), (10, 2048, 2056, 260, 4),
                   (28, 1288, 520, 17000, 6), (40, 72, 8200, 900, 4)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", FEW_TOKEN_LINES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_few_tokens_weights_by_lines(case, dtype, device):
    test_few_tokens_match_the_operators(case, dtype, device)


# T, H, I, N, k: two launches up to 16 tokens, hidden 1024 and 2^23 weights a projection (the MLP alone any hidden and 2^22), and one past each of the three; up to 48 tokens and
# 2^21, and one past either; one column group and the last of several short; fewer pairs than waves, more than two to a wave; one split of K
MERGED_LAUNCH_CASES = [(1, 1024, 4096, 4096, 16), (16, 1024, 8192, 4096, 32), (16, 1024, 8200, 4096, 16), (17, 1024, 4096, 4096, 16), (16, 1032, 4096, 4096, 16), (5, 8, 64, 64, 2),
                       (9, 520, 2056, 90000, 18), (3, 1016, 72, 260, 4), (48, 512, 4096, 1024, 8), (49, 512, 4096, 1024, 8), (48, 520, 4096, 1024, 8), (33, 1024, 2048, 4096, 16),
                       (20, 264, 520, 1000, 32), (16, 2048, 2048, 1024, 8)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", MERGED_LAUNCH_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_few_tokens_in_two_launches(case, dtype, device):
    """Against the operators; then call after call on changing inputs in the same memory, and replays of a graph with eager calls between them: every result has the bits of its
    input's first one, whoever of a token's blocks came last."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    test_few_tokens_match_the_operators(case, dtype, device)
    T, H, I, N, k = case
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device, dtype=dtype).eval()
    g = torch.Generator(device=device).manual_seed(T + H)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, H ** -0.5, generator=g)
        xs = [torch.randn(1, T, H, device=device, generator=g).to(dtype) for _ in range(4)]
        first = [layer(x).clone() for x in xs]
        mlp = [layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight]
        alone = [_ops().hip_omni_mlp_func(x[0], *mlp, residual=xs[0][0]).clone() for x in xs]
        for _ in range(20):
            again = [layer(x) for x in xs]
            assert all(torch.equal(a, b) for a, b in zip(first, again))
            again = [_ops().hip_omni_mlp_func(x[0], *mlp, residual=xs[0][0]) for x in xs]
            assert all(torch.equal(a, b) for a, b in zip(alone, again))
        held, stream = xs[0].clone(), torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            layer(held)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(held)
        for i in range(8):
            held.copy_(xs[i % 4])
            graph.replay()
            assert torch.equal(y, first[i % 4])
            assert torch.equal(layer(xs[(i + 1) % 4]), first[(i + 1) % 4])


def _few_tokens_plan(T, H, I, r, captured=False):
    """Launches, staged rows, K units at once in the first launch and the second, parts of the down projection (r 0: the MLP alone)."""
    import ctypes
    from omni_moe.ops.hip import _lib
    out = (ctypes.c_int32 * 5)()
    assert _lib.load().omni_probe_few_tokens(T, H, I, r, captured, ctypes.addressof(out)) == 0
    return tuple(out)


# T, H, I, N, k and the plan: at most eight tokens in three launches (hidden past 1024), one and two K units of a wave at once; more than eight units to a part in two launches and
# in three; 64 tokens, whose weights stay in registers, with two units at once and no K tail
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case, plan", [((1, 2048, 8192, 4096, 16), (3, 8, 2, 2, 4)), ((8, 4096, 520, 1024, 4), (3, 8, 2, 2, 1)), ((5, 1032, 4104, 576, 8), (3, 8, 2, 2, 7)),
                                        ((8, 1040, 264, 256, 8), (3, 8, 2, 1, 1)), ((8, 2048, 8200, 1000, 4), (3, 8, 2, 2, 4)), ((8, 256, 8192, 1024, 8), (2, 8, 1, 2, 8)),
                                        ((3, 264, 7944, 256, 4), (2, 8, 1, 2, 8)), ((64, 768, 8192, 256, 4), (3, 64, 1, 2, 8))], ids=str)
def test_few_tokens_on_every_plan(case, plan, dtype, device):
    T, H, I, N, _ = case
    assert _few_tokens_plan(T, H, I, int(N ** 0.5)) == plan
    test_few_tokens_match_the_operators(case, dtype, device)


# ... and of the MLP alone, which takes two launches for other sizes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case, plan", [((8, 8200, 512), (3, 8, 2, 1, 1)), ((7, 2048, 8192), (3, 8, 2, 2, 4)), ((8, 1040, 520), (2, 8, 2, 2, 1)), ((6, 512, 512), (2, 8, 1, 1, 1))], ids=str)
def test_mlp_of_few_tokens_on_every_plan(case, plan, dtype, device):
    assert _few_tokens_plan(*case, 0) == plan
    test_mlp_matches_oracle(case, dtype, device)


def _graph_nodes(call):
    """Nodes of a graph that one call is captured into: its launches."""
    import ctypes
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        y = call()
    count = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    graph.replay()
    torch.cuda.synchronize()
    return count.value, y


# T, H, I of a layer and launches when a program makes the call, when it is captured; the same for its MLP alone.  A replay has no host work, so that two launches are taken only
# where their kernels are no slower: both sides of the lines at 3 * 2^20 weights a projection, 2^21 beyond 16 tokens, 2^19 for the MLP
@pytest.mark.parametrize("case, layer, mlp", [((16, 1024, 4096), (2, 3), (2, 3)), ((16, 768, 4096), (2, 2), (2, 3)), ((5, 768, 4104), (2, 3), (2, 3)), ((48, 1024, 2048), (2, 2), (2, 3)),
                                              ((16, 512, 1024), (2, 2), (2, 2)), ((17, 512, 1024), (2, 2), (2, 3)), ((16, 520, 1024), (2, 2), (2, 3)), ((2, 2048, 4096), (3, 3), (3, 3))], ids=str)
def test_captured_calls_of_few_tokens_take_the_launches_that_replay_faster(case, layer, mlp, device):
    """... and leave the bits of the call that a program makes."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I = case
    assert tuple(_few_tokens_plan(T, H, I, 16, c)[0] for c in (False, True)) == layer
    assert tuple(_few_tokens_plan(T, H, I, 0, c)[0] for c in (False, True)) == mlp
    module = OmniMoE(OmniMoEConfig(H, I, "silu", 256, 8)).to(device=device, dtype=torch.bfloat16).eval()
    g = torch.Generator(device=device).manual_seed(T + I)
    with torch.no_grad():
        for p in module.parameters():
            p.normal_(0.0, H ** -0.5, generator=g)
        x = torch.randn(1, T, H, device=device, generator=g).bfloat16()
        alone = lambda: _ops().hip_omni_mlp_func(x[0], module.gate_proj.weight, module.up_proj.weight, module.down_proj.weight)
        for call, launches in ((lambda: module(x), layer), (alone, mlp)):
            want = call()
            nodes, y = _graph_nodes(call)
            assert nodes == launches[1]
            assert torch.equal(y, want)


# T, H, I: 32-row and 32-column tiles and their remainders, K of one to five tiles of 32 and with a remainder, more and fewer waves than K tiles
@pytest.mark.parametrize("case", [(1, 4, 4), (33, 36, 100), (512, 256, 1024), (100, 1028, 68), (640, 160, 96), (65, 128, 132),
                   # 256 and 288 blocks of the SwiGLU product (two ring stages, one), 512 and 544 of the down projection
                   (256, 160, 1024), (257, 160, 1024), (257, 32, 1024), (512, 1024, 544), (513, 1024, 544)], ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}")
def test_small_fp32_products_match_fp64(case, device):
    """Single precision with few output tiles: the MLP (SwiGLU and residual epilogues) and the router projection's column statistics against 64
    bits.  Tolerance: sums of K products in 32 bits, sqrt(K) * 2^-24 of the terms' size each, times 8."""
    T, H, I = case
    print(f"small fp32 {case}", flush=True)
    g = torch.Generator().manual_seed(T)
    x, res = torch.randn(T, H, generator=g), torch.randn(T, H, generator=g)
    wg, wu, wd = torch.randn(I, H, generator=g) * H ** -0.5, torch.randn(I, H, generator=g) * H ** -0.5, torch.randn(H, I, generator=g) * I ** -0.5
    want = oracle.mlp_forward(x.double(), wg.double(), wu.double(), wd.double())
    got = _ops().hip_omni_mlp_func(*(t.to(device) for t in (x, wg, wu, wd)), residual=res.to(device)).cpu().double()
    assert (got - (want + res.double())).abs().max().item() <= 8 * 2 ** -24 * (H ** 0.5 + I ** 0.5) * max(1.0, float(want.abs().max()))
    if T == 1:
        return
    for r in (32, 30):                                       # the halves' weights begin and end with a block, or inside one
        wx, wy = torch.randn(r, H, generator=g) * H ** -0.5, torch.randn(r, H, generator=g) * H ** -0.5
        bufs = _bn_buffers(r, torch.float32, device) + _bn_buffers(r, torch.float32, device)
        _ops().hip_omni_router_fwd_func(x.to(device), wx.to(device), wy.to(device), *bufs, 4, training=True, momentum=1.0)
        z = x.double() @ torch.cat([wx, wy]).double().t()
        mean = torch.cat([bufs[0], bufs[3]]).cpu().double()
        var = torch.cat([bufs[1], bufs[4]]).cpu().double()
        torch.testing.assert_close(mean, z.mean(0), rtol=1e-5, atol=8 * 2 ** -24 * H ** 0.5)
        torch.testing.assert_close(var, z.var(0), rtol=1e-5, atol=8 * 2 ** -24 * H ** 0.5)


# T, H, I, N, k: past the few-token launches; tile shapes and K splits change with T and H, the selection finds room beside the down projection or not,
# 2, 4 and 8 keys a lane, a key count that is not a multiple of 8 and one beyond the joint launch's registers (both on launches of their own)
JOINT_CASES = [(65, 1024, 4096, 4096, 16), (129, 256, 512, 10000, 8), (613, 1024, 4096, 4096, 16), (700, 520, 1048, 65536, 32), (300, 2048, 2056, 262144, 32),
               (1900, 1024, 4096, 1024, 4), (200, 512, 1536, 900, 6), (90, 256, 1024, 360000, 10)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", JOINT_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_joint_launches_match_the_operators(case, dtype, device):
    """Eval mode past 64 tokens: projections, selection and add in joint launches against the operators one by one.  The router's scores may round
    differently (its sums run in another order), so the expert term is compared where both chose the same experts."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = case
    print(f"joint {case} {dtype}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device, dtype=dtype).eval()
    g = torch.Generator(device=device).manual_seed(T)
    for p in layer.parameters():
        p.normal_(0.0, H ** -0.5, generator=g)
    layer.down_proj.weight.normal_(0.0, I ** -0.5, generator=g)
    for norm in (layer.router_norm_x, layer.router_norm_y):
        norm.running_mean.normal_(0.0, 0.3, generator=g)
        norm.running_var.uniform_(0.5, 2.0, generator=g)
    x = torch.randn(1, T, H, device=device, generator=g).to(dtype)
    ops = _ops()
    gates, ids = layer.route(x[0])
    experts = ops.hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, gates, ids).double()
    mlp = ops.hip_omni_mlp_func(x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight).double()
    got = layer(x)[0].double()
    eps = torch.finfo(dtype).eps
    scale = max(1.0, float((mlp + experts).abs().max()))
    row = (got - (mlp + experts)).abs().amax(dim=1)
    assert (row <= 4 * eps * scale).double().mean().item() >= 0.95          # a token with another least expert differs by that expert's share
    assert row.max().item() <= 0.5 * scale
    assert torch.equal(layer(x)[0].double(), got)
    layer.overlap_branches = False
    assert torch.equal(layer(x)[0].double(), got)
    # batch statistics: the router stage alone on equal buffers leaves the same buffers and chooses the same experts
    layer.train()
    before = [b.clone() for b in layer.buffers()]
    gates, ids = layer.route(x[0])
    after = [b.clone() for b in layer.buffers()]
    for b, v in zip(layer.buffers(), before):
        b.copy_(v)
    got = layer(x)[0].double()
    assert all(torch.equal(a, b) for a, b in zip(after, layer.buffers()))
    experts = ops.hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, gates, ids).double()
    assert (got - (mlp + experts)).abs().max().item() <= 4 * eps * max(1.0, float((mlp + experts).abs().max()))


# T, H, I, N, k: the joint projections on tiles of 256, 192 and 96 rows of 128 columns, whole and one row past them; the down projection on tiles of 64 x 64, 96 x 128 and
# 128 x 128, split along K and not (test_joint_launches_select_beside_every_tile: the others, and the selection beside each)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", [(613, 1024, 4096, 4096, 16), (97, 136, 2056, 576, 8), (192, 264, 4104, 576, 8), (385, 264, 4104, 576, 8), (768, 776, 2568, 1024, 4),
                                  (1153, 776, 2568, 576, 8), (1153, 264, 4104, 576, 6), (1200, 1024, 4096, 4096, 16), (1500, 1024, 4096, 1024, 8)],
                         ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_joint_launches_on_lower_tiles(case, dtype, device):
    test_joint_launches_match_the_operators(case, dtype, device)


# the joint projections on tiles of 64 x 64, hidden sizes on both sides of the line between two ring stages for gate and up and three
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", [(70, 1536, 3072, 1024, 8), (70, 1544, 3072, 1024, 8), (129, 2048, 1032, 576, 8)], ids=lambda c: "x".join(map(str, c)))
def test_joint_launches_on_short_and_long_sums(case, dtype, device):
    import ctypes
    import math
    from omni_moe.ops.hip import _lib
    T, H, I, N, k = case
    pair, down = (ctypes.c_int32 * 2)(), (ctypes.c_int32 * 4)()
    assert _lib.load().omni_probe_joint_tiles(T, H, I, math.isqrt(N), k, ctypes.addressof(pair), ctypes.addressof(down)) == 0
    assert tuple(pair) == (64, 64)
    test_joint_launches_match_the_operators(case, dtype, device)


# T, H, I, N, k, and rows, columns and parts of the down projection's tiles beside which the selection runs; of batch statistics the selecting blocks merge (r <= 128)
DOWN_CASES = [((950, 2048, 4096, 1024, 8), (192, 128, 2)), ((1295, 3128, 128, 64, 8), (192, 128, 1)), ((385, 2208, 7616, 4096, 8), (256, 128, 6)),
              ((805, 2048, 4096, 1024, 8), (128, 128, 1)), ((583, 520, 4096, 1024, 8), (96, 128, 5)), ((879, 520, 256, 1024, 8), (96, 128, 1)),
              ((213, 512, 4096, 1024, 8), (64, 64, 7)), ((657, 768, 1024, 1024, 8), (64, 64, 1)), ((694, 1536, 4096, 1024, 8), (128, 128, 2))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case, tiles", DOWN_CASES, ids=lambda c: "x".join(map(str, c)))
def test_joint_launches_select_beside_every_tile(case, tiles, dtype, device):
    """The rule's choice is asked for first, so that figures fitted anew cannot take a kernel out of the test unnoticed."""
    import ctypes
    import math
    from omni_moe.ops.hip import _lib
    T, H, I, N, k = case
    pair, down = (ctypes.c_int32 * 2)(), (ctypes.c_int32 * 4)()
    assert _lib.load().omni_probe_joint_tiles(T, H, I, math.isqrt(N), k, ctypes.addressof(pair), ctypes.addressof(down)) == 0
    assert tuple(down) == (*tiles, 1)
    test_joint_launches_match_the_operators(case, dtype, device)


# down projections in parts because the experts' kernel adds them up: few row tiles, a short one at the end, K in whole steps of a split and not, the most parts and two
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case, tiles", [((613, 1024, 4096, 4096, 16), (96, 128, 3)), ((197, 512, 1536, 576, 4), (64, 64, 6)), ((221, 1024, 2048, 6400, 8), (64, 64, 3)),
                                         ((207, 1536, 3072, 7744, 16), (64, 64, 2)), ((85, 256, 1024, 3136, 8), (64, 64, 4))], ids=lambda c: "x".join(map(str, c)))
def test_joint_launches_down_in_parts(case, tiles, dtype, device):
    test_joint_launches_select_beside_every_tile(case, tiles, dtype, device)



def test_layer_with_rows_beyond_the_tile_kernels_reach(device):
    """An intermediate size whose rows put 256 of them beyond 2 GiB: no joint launch, and the result of the operators one by one (MLP in 64 bits)."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = 65, 8, 4194312, 64, 2
    print(f"layer T={T} H={H} I={I}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device, dtype=torch.bfloat16).eval()
    g = torch.Generator(device=device).manual_seed(7)
    for p in layer.parameters():
        p.normal_(0.0, p.size(1) ** -0.5, generator=g)
    x = torch.randn(1, T, H, device=device, generator=g).bfloat16()
    got = layer(x)[0].double()
    experts = _ops().hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, *layer.route(x[0])).double()
    xd, wg, wu, wd = (t.double() for t in (x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight))
    h = (torch.nn.functional.silu((xd @ wg.t()).bfloat16().double()) * (xd @ wu.t()).bfloat16().double()).bfloat16().double()
    want = h @ wd.t() + experts
    # h rounds alike but for last bits here and there; the sum of 4 million products runs in 32 bits, over partial sums of one wave each
    assert (got - want).abs().max().item() <= 4 * 2.0 ** -7 * max(1.0, want.abs().max().item())


# T, H, I, N, k
GATHER_BY_NAME_CASES = [(300, 1024, 2048, 1024, 32), (1000, 512, 1024, 4096, 34), (512, 2048, 2048, 1024, 16), (257, 1024, 1024, 1024, 8)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("case", GATHER_BY_NAME_CASES, ids=lambda c: f"T{c[0]}-H{c[1]}-I{c[2]}-N{c[3]}-k{c[4]}")
def test_layer_gather_by_name_is_the_operator(case, dtype, device):
    """The gather algorithm by name adds a token's slots one after the other, in the joint launches' last kernel as in the operator.  An MLP of zeros leaves the
    experts' rows alone in the output; batch statistics, where the joint launches choose the router stage's experts with its gates."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    T, H, I, N, k = case
    print(f"gather by name {case} {dtype}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", N, k)).to(device=device, dtype=dtype)
    layer.expert_algo = "gather"
    g = torch.Generator(device=device).manual_seed(T)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, H ** -0.5, generator=g)
        layer.down_proj.weight.zero_()
        x = torch.randn(1, T, H, device=device, generator=g).to(dtype)
        gates, ids = layer.route(x[0])
        got = layer(x)[0]
    want = _ops().hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, gates, ids, algo="gather")
    assert torch.equal(got, want)


# one strip, ragged strips, the most strips a block merges at 64 keys and one more, 8 to 128 keys; 136 keys: the merge's own launch; top-56 and up: a selection that
# does not fit beside the down projection's tiles, behind the merge's own launch
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("case", [(2, 8), (33, 64), (700, 104), (2048, 128), (4096, 64), (4100, 64), (300, 136), (700, 64, 64), (2048, 24, 56), (3, 16, 128)],
                         ids=lambda c: ("T%d-r%d" if len(c) == 2 else "T%d-r%d-k%d") % c)
def test_joint_batch_statistics_equal_the_router_stage(case, dtype, device):
    """A small layer merges the batch statistics inside its joint launches: buffers and counts as the router stage (which launches the merge) leaves them on the
    same input, to the last bit of an fp32 result (double sums in another order) rounded to the buffers' type."""
    from omni_moe.modules.omni_moe import OmniMoE, OmniMoEConfig
    from omni_moe.ops import hip
    T, r, k = (*case, 8)[:3]
    H, I = 64, 128
    print(f"joint statistics T={T} r={r} k={k} {dtype}", flush=True)
    layer = OmniMoE(OmniMoEConfig(H, I, "silu", r * r, k)).to(device=device, dtype=dtype)
    g = torch.Generator(device=device).manual_seed(T + r)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05, generator=g)
        for n in (layer.router_norm_x, layer.router_norm_y):
            n.running_mean.normal_(0.0, 0.3, generator=g)
            n.running_var.uniform_(0.5, 1.5, generator=g)
        x = torch.empty(1, T, H, device=device, dtype=dtype).normal_(0.0, 1.0, generator=g)
        stats = [b.clone() for n in (layer.router_norm_x, layer.router_norm_y) for b in (n.running_mean, n.running_var, n.num_batches_tracked)]
        gates, ids = hip.hip_omni_router_fwd_func(x[0], layer.router_gate_x.weight, layer.router_gate_y.weight, *stats, k, training=True)
        y = layer(x)
        if k > 8 and dtype != torch.float32:                               # both merge in a launch of its own: the same choice, to the bit
            experts = hip.hip_omni_expert_func(x[0], layer.up_embed.weight, layer.down_embed.weight, gates, ids)
            want = hip.hip_omni_mlp_func(x[0], layer.gate_proj.weight, layer.up_proj.weight, layer.down_proj.weight).float() + experts.float()
            # sums of the same terms in another order, a rounding at each of three places
            assert ((y[0].float() - want).abs() <= 4 * {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype] * want.abs().max()).all()
    got = [b for n in (layer.router_norm_x, layer.router_norm_y) for b in (n.running_mean, n.running_var, n.num_batches_tracked)]
    ulp = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -22}[dtype]      # neighbours of the buffers' type
    for a, b in zip(got, stats):
        if a.dtype == torch.int64:
            assert torch.equal(a, b)
        else:
            assert ((a.float() - b.float()).abs() <= 1.01 * ulp * b.float().abs() + 1e-6).all()     # 1e-6: where the two terms of the moving average cancel
