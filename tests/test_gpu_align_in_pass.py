"""Calls whose gate-up pass aligns the ids itself: the bits of the steps, at the edges of what it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

_BF, _FP = torch.bfloat16, torch.float16
_CASES = [  # T, E, K, H, I, dtype, layout, activation, bias
    (17, 128, 8, 256, 128, _BF, "tiled", "silu", False),
    (128, 128, 8, 256, 128, _BF, "plain", "silu", False),       # 1024 ids, the most
    (129, 128, 8, 256, 128, _BF, "plain", "silu", False),       # one token more: aligned in front
    (500, 3, 2, 96, 64, _FP, "plain", "silu", False),           # long runs of an expert's blocks, a tail unit
    (341, 256, 3, 128, 64, _BF, "plain", "swigluoai", True),    # most experts
    (33, 40, 6, 160, 96, _FP, "plain", "gelu", False),          # experts that are no power of two
    (64, 1, 1, 128, 128, _BF, "plain", "silu", False),          # one expert
    (100, 128, 8, 512, 384, "e4m3", "plain", "silu", False),
    (40, 64, 4, 160, 96, "e4m3", "plain", "silu", False),
]


@pytest.mark.parametrize("case", _CASES, ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
@pytest.mark.parametrize("given", [False, True])
def test_bits_of_the_steps(moe, dev, monkeypatch, case, given):
    print(case, given, flush=True)
    T, E, K, H, I, dtype, layout, activation, bias = case
    g = torch.Generator().manual_seed(T + E + H)
    draw = lambda *shape, std=1.0: torch.randn(*shape, generator=g) * std
    act = _BF if dtype == "e4m3" else dtype
    x, logits = draw(T, H).to(act).to(dev), (draw(T, E) + 2 * draw(E)).to(act).to(dev)
    w13, w2 = draw(E, 2 * I, H, std=0.1).to(act).to(dev), draw(E, H, I, std=0.1).to(act).to(dev)
    kw = dict(activation=activation)
    if bias:
        kw.update(w1_bias=draw(E, 2 * I, std=0.1).to(act).to(dev), w2_bias=draw(E, H, std=0.1).to(act).to(dev))
    if layout == "tiled":
        w13, w2 = moe.ops.tile_expert_weights(w13, True, False), moe.ops.tile_expert_weights(w2, False)
        kw["weight_layout"] = "tiled"
    if dtype == "e4m3":
        w13, s13, w2, s2 = moe.quantize_expert_weights(w13, w2)
        kw.update(w1_scale=s13, w2_scale=s2)
    if given:
        tw, ids, _ = moe.fused_topk(x, logits, K, True)
        b13, b2 = kw.pop("w1_bias", None), kw.pop("w2_bias", None)
        call = lambda: moe.fused_experts(x, w13, w2, b13, b2, tw, ids, **kw)
    else:
        call = lambda: moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    for _ in range(3):   # (other calls' workspaces in between)
        one = call()
        torch.empty(1 << 20, device=dev).fill_(float("nan"))
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = call()
    assert bool(steps.isfinite().all()) and float(steps.float().abs().max()) > 0 and torch.equal(one, steps)


@pytest.mark.parametrize("T", [100, 700])   # aligned in the pass; by a workgroup for every 1024 ids
def test_replay_from_a_graph(moe, dev, T):
    E, K, H, I = 64, 8, 256, 128
    g = torch.Generator().manual_seed(T)
    x, logits = torch.randn(T, H, generator=g).to(_BF).to(dev), torch.randn(T, E, generator=g).to(_BF).to(dev)
    w13 = (0.1 * torch.randn(E, 2 * I, H, generator=g)).to(_BF).to(dev)
    w2 = (0.1 * torch.randn(E, H, I, generator=g)).to(_BF).to(dev)
    moe.fused_topk_experts(x, logits, w13, w2, K, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = moe.fused_topk_experts(x, logits, w13, w2, K, True)
    for _ in range(4):
        x.normal_()
        logits.normal_()
        graph.replay()
        assert torch.equal(out, moe.fused_topk_experts(x, logits, w13, w2, K, True))
        torch.cuda.synchronize()
