"""e4m3 down pass that quantises its tokens itself: the bits of the quantisation in a launch of its own, which calls with a
bias (here of zero) keep, at every row length it serves and on both sides of its line, few and many blocks a share, blocks that
are full and hardly filled."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _codes_of_the_intermediate(moe, ws, x, E, K, I):
    """Where in the workspace of a call with blocks of 32 a launch in front of the down pass leaves the intermediate's codes."""
    T, H = x.shape
    up = lambda n: -(-n // 256) * 256
    rows = -(-(T * K + 31 * E) // 32) * 32
    start = up(rows * I * 2) + up(T * K * H * 2) + up(T * H) + up(T * 4)
    return ws[start:start + rows * I]


def _workspace(moe, x, E, K, I):
    code = moe._lib.DTYPE_CODE[x.dtype]
    size = moe._lib.lib().moe_fused_experts_workspace_bytes(x.size(0), x.size(1), I, E, K, 32, code, moe._lib.E4M3_CODE)
    return torch.full((size,), 0xA5, dtype=torch.uint8, device=x.device)


@pytest.mark.parametrize("T,E,K,H,I,dtype,on_input,in_pass", [
    (300, 4, 2, 16, 384, "bfloat16", False, True),   # one group a block, more blocks than experts
    (2000, 8, 4, 16, 768, "float16", False, False),
    (300, 8, 2, 32, 512, "bfloat16", True, False),   # two groups, three
    (500, 8, 2, 48, 768, "bfloat16", False, False),
    (64, 4, 2, 64, 384, "bfloat16", False, True),   # the fewest ids; four groups of rows a block, fewer than there are shares
    (16, 16, 8, 160, 512, "float16", False, False),   # ten groups a block: wavefronts without one
    (43, 32, 3, 2048, 768, "bfloat16", False, False),   # (a small share of long rows: codes of a launch)
    (100, 128, 8, 2048, 768, "bfloat16", True, True),
    (300, 8, 2, 1024, 384, "float16", True, True),   # experts of several blocks
    (3000, 5, 2, 96, 512, "bfloat16", False, False),    # many blocks a share, six groups each
    (2500, 3, 1, 288, 768, "float16", False, False),
    (1200, 16, 4, 64, 384, "bfloat16", False, True),
    (64, 4, 2, 64, 128, "float16", False, True),   # rows of one unit: a ring of one place
    (900, 8, 2, 272, 128, "bfloat16", True, True),
    (100, 64, 4, 1024, 256, "bfloat16", False, True),
    (1100, 6, 2, 48, 256, "float16", False, True),
    (300, 64, 4, 1024, 640, "float16", False, True),   # an odd number of units
    (2500, 8, 4, 160, 640, "bfloat16", True, True),
    (2750, 3, 2, 288, 512, "float16", False, True),    # rows that two pairs a wavefront code, in many blocks of few groups
    (8250, 8, 4, 48, 768, "bfloat16", False, True),
    (25000, 8, 4, 16, 512, "bfloat16", False, True),   # and of one
    (130, 32, 4, 2048, 768, "float16", True, True),    # the least share of such rows, and less
    (127, 32, 4, 2048, 768, "float16", True, False),
])
def test_codes_made_in_the_down_pass_have_the_bits_of_the_launch(moe, dev, T, E, K, H, I, dtype, on_input, in_pass):
    print(T, E, K, H, I, dtype, on_input, in_pass, flush=True)
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
        out, ws = torch.full_like(x, float("nan")), _workspace(moe, x, E, K, I)
        fm.launch_fused_experts(x, out, q13, q2, None, b2, s13, s2, tw, so, eo, npp, 32, "silu", on_input,
                                weight_code=moe._lib.E4M3_CODE, workspace=ws)
        assert bool((_codes_of_the_intermediate(moe, ws, x, E, K, I) == 0xA5).all()) == (in_pass and b2 is None)   # (who made the codes)
        return out

    want = run(torch.zeros(E, H, dtype=dt, device=dev))
    assert bool(want.isfinite().all()) and float(want.float().abs().max()) > 0
    for _ in range(2):
        assert torch.equal(run(None), want)


@pytest.mark.parametrize("T,E,H,I,in_pass", [
    (127, 4, 64, 256, False), (128, 4, 64, 256, True), (128, 4, 64, 384, True), (128, 4, 64, 64, False), (128, 4, 64, 192, False),
    (128, 4, 64, 512, False), (511, 32, 2048, 512, False), (512, 32, 2048, 512, True), (512, 32, 2048, 640, True),
    (512, 32, 2048, 768, True), (512, 32, 2032, 768, False), (2048, 32, 2048, 896, False)])
def test_which_calls_make_their_codes_in_the_down_pass(moe, dev, T, E, H, I, in_pass):
    print(T, E, H, I, flush=True)
    g = torch.Generator(dev).manual_seed(T + I)
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).bfloat16()
    x, out = draw(T, H), torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    q13, s13, q2, s2 = moe.quantize_expert_weights(draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05))
    tw, ids, _ = moe.fused_topk(x, draw(T, E), 1, False)
    so, eo, npp = moe.fused_moe.moe_align_block_size(ids, 32, E)
    ws = _workspace(moe, x, E, 1, I)
    moe.fused_moe.launch_fused_experts(x, out, q13, q2, None, None, s13, s2, tw, so, eo, npp, 32,
                                       weight_code=moe._lib.E4M3_CODE, workspace=ws)
    assert bool((_codes_of_the_intermediate(moe, ws, x, E, 1, I) == 0xA5).all()) == in_pass


def test_blocks_of_no_expert_in_a_callers_alignment(moe, dev):
    """Blocks without slots that name no expert (-1), in front of, between and behind the experts' own, change nothing."""
    g = torch.Generator(dev).manual_seed(3)
    T, E, H, I = 128, 4, 64, 384
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
        out, ws = torch.full_like(x, float("nan")), _workspace(moe, x, E, 1, I)
        moe.fused_moe.launch_fused_experts(x, out, q13, q2, None, None, s13, s2, tw, so.to(dev), eo.to(dev), npp.to(dev), 32,
                                           weight_code=moe._lib.E4M3_CODE, workspace=ws)
        assert bool((_codes_of_the_intermediate(moe, ws, x, E, 1, I) == 0xA5).all())
        return out

    want = run([0, 1, 2, 3])
    assert bool(want.isfinite().all())
    assert torch.equal(run([-1, 0, 1, -1, 2, 3, -1]), want)


def test_codes_made_in_the_down_pass_inside_a_hip_graph(moe, dev):
    g = torch.Generator(dev).manual_seed(9)
    T, E, K, H, I = 100, 64, 4, 1024, 384
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).bfloat16()
    q13, s13, q2, s2 = moe.quantize_expert_weights(draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05))
    x, logits = draw(T, H), draw(T, E)
    run = lambda: moe.fused_topk_experts(x, logits, q13, q2, K, True, w1_scale=s13, w2_scale=s2)

    def steps():   # (with a bias: the codes of a launch)
        tw, ids, _ = moe.fused_topk(x, logits, K, True)
        so, eo, npp = moe.fused_moe.moe_align_block_size(ids, 32, E)
        out = torch.empty_like(x)
        moe.fused_moe.launch_fused_experts(x, out, q13, q2, None, torch.zeros_like(q2[:, :, 0], dtype=x.dtype), s13, s2, tw, so,
                                           eo, npp, 32, weight_code=moe._lib.E4M3_CODE)
        return out

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
        assert torch.equal(captured, run()) and torch.equal(captured, steps())
