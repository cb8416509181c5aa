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


@pytest.mark.parametrize("T,E,K,H,dtype,kind", [(100, 64, 8, 256, _BF, "holes"), (512, 5, 2, 160, _FP, "holes"),
                                                (128, 256, 8, 256, "e4m3", "holes"), (40, 16, 4, 256, _BF, "none"),
                                                (40, 16, 4, 256, "e4m3", "none"), (1, 1, 1, 128, _BF, "all")])
def test_given_ids_that_are_no_experts(moe, dev, monkeypatch, T, E, K, H, dtype, kind):
    """Ids out of range are left out: the alignment that the pass leaves in the layer's workspace is that of the alignment
    kernels, and tokens whose ids are all experts' have the bits of the steps."""
    print(T, E, K, H, dtype, kind, flush=True)
    I, act, lib = 128, _BF if dtype == "e4m3" else dtype, moe._lib
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, H, generator=g).to(act).to(dev)
    w13, w2 = ((0.1 * torch.randn(*s, generator=g)).to(act).to(dev) for s in ((E, 2 * I, H), (E, H, I)))
    ids = torch.randint(0, E, (T, K), generator=g, dtype=torch.int32)
    if kind == "holes":
        bad = torch.rand(T, 1, generator=g) < 0.4
        ids = torch.where(bad & (torch.rand(T, K, generator=g) < 0.5), torch.where(torch.rand(T, K, generator=g) < 0.5, -1, E), ids).int()
    elif kind == "none":
        ids.fill_(E)
    tw, ids, s13, s2 = torch.rand(T, K, generator=g).to(dev), ids.to(dev), None, None
    if dtype == "e4m3":
        w13, s13, w2, s2 = moe.quantize_expert_weights(w13, w2)
    out, ptr = torch.empty_like(x), lambda t: None if t is None else t.data_ptr()
    code = lib.DTYPE_CODE[act]
    args = lib.MoeLayerArgs(x=ptr(x), out=ptr(out), w13=ptr(w13), w2=ptr(w2), w13_scale=ptr(s13), w2_scale=ptr(s2),
                            topk_weights=ptr(tw), topk_ids=ptr(ids), w13_stride_e=w13.stride(0), w13_stride_n=w13.stride(1),
                            w2_stride_e=w2.stride(0), w2_stride_n=w2.stride(1), T=T, H=H, I=I, E=E, K=K, act_dtype=code,
                            weight_dtype=code if s13 is None else lib.E4M3_CODE, swiglu_alpha=1.702, swiglu_limit=7.0,
                            stream=torch.cuda.current_stream(dev).cuda_stream)
    size = lib.lib().moe_layer_workspace_bytes(args)
    ws = torch.full((size,), 0x5a, dtype=torch.uint8, device=dev)
    args.workspace, args.workspace_bytes = ws.data_ptr(), size
    lib.check(lib.lib().moe_layer(args))
    # the workspace of a call whose ids are given starts with the sorted slots, the blocks' experts and the padded count
    at, got = 0, []
    want = moe.moe_align_block_size(ids, 32, E)
    for t in want:
        got.append(ws[at:at + 4 * t.numel()].clone().view(torch.int32))
        at += (4 * t.numel() + 255) // 256 * 256
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = moe.fused_experts(x, w13, w2, None, None, tw, ids, w1_scale=s13, w2_scale=s2)
    whole = ((ids >= 0) & (ids < E)).all(1)
    assert bool(whole.any()) == (kind != "none") and torch.equal(out[whole], steps[whole])
    assert bool(steps[whole].isfinite().all())
