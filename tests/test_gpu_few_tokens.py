"""The layer call of a few tokens in two launches: the bits of the steps it replaces, at the edges of what it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _args(moe, dev, T, E, K, H, I, dtype, layout, activation, bias, on_input, logits_dtype):
    g = torch.Generator().manual_seed(T + 7 * E + H + I)
    draw = lambda *shape, std=1.0: torch.randn(*shape, generator=g) * std
    x, logits = draw(T, H).to(dtype).to(dev), (draw(T, E) + 2 * draw(E)).to(logits_dtype).to(dev)
    w13, w2 = draw(E, 2 * I, H, std=0.05).to(dtype).to(dev), draw(E, H, I, std=0.05).to(dtype).to(dev)
    kw = dict(activation=activation, apply_router_weight_on_input=on_input)
    if bias:
        kw.update(w1_bias=draw(E, 2 * I, std=0.1).to(dtype).to(dev), w2_bias=draw(E, H, std=0.1).to(dtype).to(dev))
    if layout == "tiled":
        w13 = moe.ops.tile_expert_weights(w13, True, activation == "swigluoai")
        w2, kw["weight_layout"] = moe.ops.tile_expert_weights(w2, False), "tiled"
    if layout == "strided":   # rows further apart than their length, in a buffer of neighbours that must not be read as weights
        w13 = torch.cat([w13, torch.full_like(w13[:, :, :64], 50.0)], 2)[:, :, :H]
        w2 = torch.cat([w2, torch.full_like(w2[:, :, :64], 50.0)], 2)[:, :, :I]
    return x, logits, w13, w2, K, kw


_BF, _FP, _F32 = torch.bfloat16, torch.float16, torch.float32
_CASES = [  # T, E, K, H, I, dtype, layout, activation, bias, on_input, logits dtype
    (1, 128, 8, 512, 384, _BF, "plain", "silu", False, False, _BF),       # the fewest steps a pass has
    (1, 32, 1, 320, 320, _FP, "plain", "silu", False, False, _FP),        # an odd number of them
    (2, 64, 2, 1024, 384, _BF, "tiled", "silu", False, False, _F32),
    (3, 256, 8, 512, 384, _FP, "tiled", "gelu", False, False, _FP),
    (7, 32, 4, 2880, 320, _BF, "plain", "swigluoai", True, False, _BF),   # two workgroups of the down pass a CU
    (8, 64, 8, 4096, 384, _BF, "strided", "silu", True, False, _BF),      # most hidden states
    (9, 32, 6, 640, 448, _FP, "strided", "silu", False, True, _BF),
    (12, 128, 8, 2048, 768, _BF, "plain", "silu", False, False, _BF),     # most (token, k)
    (13, 128, 8, 512, 384, _BF, "plain", "silu", False, False, _BF),      # one token more: the steps
    (16, 32, 6, 512, 384, _BF, "tiled", "swigluoai", True, True, _BF),    # most tokens, several to an expert
    (16, 256, 2, 512, 512, _FP, "plain", "gelu", True, False, _F32),
]


@pytest.mark.parametrize("case", _CASES, ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
def test_few_tokens_have_the_bits_of_the_steps(moe, dev, monkeypatch, case):
    print(case, flush=True)
    x, logits, w13, w2, K, kw = _args(moe, dev, *case)
    one = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    again = moe.fused_topk_experts(x, logits, w13, w2, K, False, **kw)
    inplace = x.clone()
    assert moe.fused_topk_experts(inplace, logits, w13, w2, K, True, inplace=True, **kw) is inplace
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    assert bool(steps.isfinite().all()) and float(steps.float().abs().max()) > 0
    assert torch.equal(one, steps) and torch.equal(inplace, steps)
    assert torch.equal(again, moe.fused_topk_experts(x, logits, w13, w2, K, False, **kw))


def test_all_tokens_on_the_same_experts_and_rows_that_are_no_numbers(moe, dev, monkeypatch):
    """Experts with all sixteen tokens, whose columns take two passes; and logits of NaN, whose ids repeat: those rows are
    NaN, as the steps have them, and the others are not touched."""
    x, logits, w13, w2, K, kw = _args(moe, dev, 16, 32, 6, 512, 384, _BF, "plain", "silu", False, False, _BF)
    logits = logits[:1].expand(16, 32).contiguous()
    lost = logits.clone()
    lost[3], lost[11] = float("nan"), float("nan")
    got = [moe.fused_topk_experts(x, l, w13, w2, K, True) for l in (logits, lost)]
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    want = moe.fused_topk_experts(x, logits, w13, w2, K, True)
    assert torch.equal(got[0], want)
    rows = torch.ones(16, dtype=torch.bool, device=dev)
    rows[3] = rows[11] = False
    assert torch.equal(got[1][rows], want[rows]) and bool(got[1][~rows].isnan().all())


@pytest.mark.parametrize("activation", ["silu", "swigluoai", "gelu"])
@pytest.mark.parametrize("on_input", [False, True])
@pytest.mark.parametrize("renormalize", [False, True])
def test_rows_whose_ids_repeat_have_every_term(moe, dev, monkeypatch, activation, on_input, renormalize):
    """Logits without a largest one go to expert 0 K times, with the weights NaN, -10000, -10000, ...: the result is that of
    the steps, whatever an earlier call (of finite rows, twice as large) left in the workspace."""
    print(activation, on_input, renormalize, flush=True)
    x, logits, w13, w2, K, kw = _args(moe, dev, 12, 32, 6, 512, 384, _BF, "plain", activation, False, on_input, _BF)
    lost = logits.clone()
    lost[3], lost[5, 7], lost[8], lost[11, 31] = float("nan"), float("inf"), -float("inf"), float("nan")
    got = []
    for _ in range(4):
        assert bool(moe.fused_topk_experts(2 * x, logits, w13, w2, K, renormalize, **kw).isfinite().all())
        got.append(moe.fused_topk_experts(x, lost, w13, w2, K, renormalize, **kw))
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    want = moe.fused_topk_experts(x, lost, w13, w2, K, renormalize, **kw)
    whole = torch.tensor([t not in (3, 5, 8, 11) for t in range(12)], device=dev)
    assert bool(want[whole].isfinite().all())
    for g in got:
        assert torch.equal(g.isnan(), want.isnan()) and torch.equal(g.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0))


def test_few_tokens_replay_from_a_graph(moe, dev):
    x, logits, w13, w2, K, kw = _args(moe, dev, 5, 64, 4, 512, 384, _BF, "plain", "silu", False, False, _BF)
    want = moe.fused_topk_experts(x, logits, w13, w2, K, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = moe.fused_topk_experts(x, logits, w13, w2, K, True)
    for i in range(3):
        x.normal_()
        logits.normal_()
        graph.replay()
        assert torch.equal(out, moe.fused_topk_experts(x, logits, w13, w2, K, True)) and not torch.equal(out, want)
        torch.cuda.synchronize()


@pytest.mark.parametrize("case", [
    (7, 256, 8, 4096, 384, _BF, "plain", "silu", False, False, _BF),      # most hidden states beside twelve wavefronts' rings
    (16, 32, 6, 512, 1024, _BF, "plain", "silu", False, False, _BF),      # more units to a CU than those have
    (14, 32, 6, 576, 832, _FP, "plain", "swigluoai", True, False, _BF),   # 13 of them, an odd number of steps
], ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
def test_units_of_a_cu_over_twelve_wavefronts(moe, dev, monkeypatch, case):
    print(case, flush=True)
    x, logits, w13, w2, K, kw = _args(moe, dev, *case)
    one = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    assert bool(steps.isfinite().all()) and float(steps.float().abs().max()) > 0 and torch.equal(one, steps)
