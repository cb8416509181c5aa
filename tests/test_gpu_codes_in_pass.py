"""e4m3 down pass that quantises its tokens itself: the bits of the quantisation in a launch of its own, which calls with a
bias (here of zero) keep, at every row length it serves, few and many blocks a share, blocks that are full and hardly filled."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,H,I,dtype,on_input", [
    (300, 4, 2, 16, 384, "bfloat16", False),     # one group a block, more blocks than experts
    (2000, 8, 4, 16, 768, "float16", False),
    (300, 8, 2, 32, 512, "bfloat16", True),      # two groups, three
    (500, 8, 2, 48, 768, "bfloat16", False),
    (64, 4, 2, 64, 384, "bfloat16", False),      # the fewest ids; four groups of rows a block, fewer than there are shares
    (16, 16, 8, 160, 512, "float16", False),     # ten groups a block: wavefronts without one
    (43, 32, 3, 2048, 768, "bfloat16", False),   # just beyond the line; shares that cross blocks
    (100, 128, 8, 2048, 768, "bfloat16", True),
    (300, 8, 2, 1024, 384, "float16", True),     # experts of several blocks
    (3000, 5, 2, 96, 512, "bfloat16", False),    # many blocks a share, six groups each
    (2500, 3, 1, 288, 768, "float16", False),
    (1200, 16, 4, 64, 384, "bfloat16", False),
])
def test_codes_made_in_the_down_pass_have_the_bits_of_the_launch(moe, dev, T, E, K, H, I, dtype, on_input):
    print(T, E, K, H, I, dtype, on_input, flush=True)
    fm = moe.fused_moe
    dt = getattr(torch, dtype)
    g = torch.Generator(dev).manual_seed(T + E + H)
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).to(dt)
    x = draw(T, H)
    x[T // 2] = 0   # rows of the intermediate whose scale is 1
    q13, s13, q2, s2 = moe.quantize_expert_weights(draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05))
    logits = torch.randn(T, E, generator=g, device=dev) + 2.0 * torch.rand(E, generator=g, device=dev)
    tw, ids, _ = moe.fused_topk(x, logits, K, True)
    so, eo, npp = fm.moe_align_block_size(ids, 32, E)

    def run(b2):
        out = torch.full_like(x, float("nan"))
        fm.launch_fused_experts(x, out, q13, q2, None, b2, s13, s2, tw, so, eo, npp, 32, "silu", on_input,
                                weight_code=moe._lib.E4M3_CODE)
        return out

    want = run(torch.zeros(E, H, dtype=dt, device=dev))
    assert bool(want.isfinite().all()) and float(want.float().abs().max()) > 0
    for _ in range(2):
        assert torch.equal(run(None), want)


def test_blocks_of_no_expert_in_a_callers_alignment(moe, dev):
    """Blocks without slots that name no expert (-1), in front of, between and behind the experts' own, change nothing."""
    g = torch.Generator(dev).manual_seed(3)
    T, E, H, I = 128, 4, 64, 512
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).bfloat16()
    x = draw(T, H)
    q13, s13, q2, s2 = moe.quantize_expert_weights(draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05))
    tw = torch.rand(T, 1, generator=g, device=dev)
    slots = [[t for t in range(T) if t % E == e] for e in range(E)]   # a block an expert, all of it slots

    def run(blocks):
        so = torch.full((T + E * 31,), T, dtype=torch.int32)
        for i, e in enumerate(blocks):
            if e >= 0:
                so[32 * i: 32 * i + 32] = torch.tensor(slots[e], dtype=torch.int32)
        eo = torch.full((-(-so.numel() // 32),), -1, dtype=torch.int32)
        eo[: len(blocks)] = torch.tensor(blocks, dtype=torch.int32)
        npp = torch.tensor([32 * len(blocks)], dtype=torch.int32)
        out = torch.full_like(x, float("nan"))
        moe.fused_moe.launch_fused_experts(x, out, q13, q2, None, None, s13, s2, tw, so.to(dev), eo.to(dev), npp.to(dev), 32,
                                           weight_code=moe._lib.E4M3_CODE)
        return out

    want = run([0, 1, 2, 3])
    assert bool(want.isfinite().all())
    assert torch.equal(run([-1, 0, 1, -1, 2, 3, -1]), want)


def test_codes_made_in_the_down_pass_inside_a_hip_graph(moe, dev):
    g = torch.Generator(dev).manual_seed(9)
    T, E, K, H, I = 100, 64, 4, 1024, 768
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).bfloat16()
    q13, s13, q2, s2 = moe.quantize_expert_weights(draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05))
    x, logits = draw(T, H), draw(T, E)
    run = lambda: moe.fused_topk_experts(x, logits, q13, q2, K, True, w1_scale=s13, w2_scale=s2)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = run()
    for seed in range(4):
        x.copy_(draw(T, H))
        logits.copy_(draw(T, E))
        captured.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, run())
