"""Down pass of a large call, two n-tiles of a full block a workgroup: the bits of one tile a workgroup (which calls with
biases keep, here of zero), over the fewest K tiles, odd numbers of n-tiles, blocks that are full, nearly and hardly filled."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _args(moe, dev, T, E, K, H, I, dtype, tiled, skew):
    g = torch.Generator(dev).manual_seed(T + H + I)
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).to(dtype)
    x, w13, w2 = draw(T, H), draw(E, 2 * I, H, std=0.03), draw(E, H, I, std=0.05)
    logits = torch.randn(T, E, generator=g, device=dev) + skew * torch.arange(E, device=dev)
    kw = {}
    if tiled:
        w13, w2 = moe.ops.tile_expert_weights(w13, True), moe.ops.tile_expert_weights(w2, False)
        kw["weight_layout"] = "tiled"
    tw, ids, _ = moe.fused_topk(x, logits, K, True)
    return x, w13, w2, tw, ids, kw


_CASES = [  # T, E, K, H, I, dtype, tiled, skew
    (7600, 4, 2, 4096, 128, torch.bfloat16, False, 0.3),   # two K tiles: the fewest
    (7600, 4, 2, 4096, 256, torch.float16, True, 0.0),
    (17200, 8, 2, 1792, 192, torch.bfloat16, False, 0.5),  # seven n-tiles: the last of a block has no partner
    (8192, 1, 1, 8192, 128, torch.bfloat16, False, 0.0),   # every block full
    (30720, 3, 1, 2048, 320, torch.float16, False, 0.0),
]


@pytest.mark.parametrize("T,E,K,H,I,dtype,tiled,skew", _CASES)
def test_two_tiles_a_workgroup_have_the_bits_of_one(moe, dev, T, E, K, H, I, dtype, tiled, skew):
    print(T, E, K, H, I, dtype, tiled, flush=True)
    x, w13, w2, tw, ids, kw = _args(moe, dev, T, E, K, H, I, dtype, tiled, skew)
    b13, b2 = torch.zeros(E, 2 * I, dtype=dtype, device=dev), torch.zeros(E, H, dtype=dtype, device=dev)
    want = moe.fused_experts(x, w13, w2, b13, b2, tw, ids, **kw)
    assert bool(want.isfinite().all()) and float(want.float().abs().max()) > 0
    for _ in range(3):
        assert torch.equal(moe.fused_experts(x, w13, w2, None, None, tw, ids, **kw), want)


@pytest.mark.parametrize("T,E,K,H,I,on_input", [
    (26000, 4, 1, 4096, 256, False),
    (29200, 4, 2, 1792, 256, False),   # seven n-tiles: the last of a block has no partner
    (26000, 4, 1, 4096, 256, True),
])
def test_e4m3_tiles_in_pairs_against_smaller_calls(moe, dev, T, E, K, H, I, on_input):
    """e4m3 takes no biases: the same rows in calls below the line."""
    print(T, E, K, H, I, on_input, flush=True)
    x, w13, w2, tw, ids, _ = _args(moe, dev, T, E, K, H, I, torch.bfloat16, False, 0.2)
    q13, s13, q2, s2 = moe.quantize_expert_weights(w13, w2)
    run = lambda a, b: moe.fused_experts(x[a:b], q13, q2, None, None, tw[a:b], ids[a:b], w1_scale=s13, w2_scale=s2,
                                         apply_router_weight_on_input=on_input)
    whole = run(0, T)
    assert bool(whole.isfinite().all()) and float(whole.float().abs().max()) > 0
    part = T // 4
    assert moe._lib.lib().moe_call_block_size(part, H, I, E, K, 2, 3, 0) == 256
    parts = torch.cat([run(a, a + part) for a in range(0, T, part)])
    assert torch.equal(whole, parts)


@pytest.mark.parametrize("T,E,K,H,I,dtype,tiled,skew", [_CASES[0], _CASES[1], _CASES[2]])
@pytest.mark.parametrize("on_input", [False, True])
def test_pairs_in_launches_of_their_own_and_across_xcds(moe, dev, T, E, K, H, I, dtype, tiled, skew, on_input):
    """The passes as two launches, one by one, and as one whose every hand-off crosses XCDs: the bits of one tile a workgroup."""
    print(T, E, K, H, I, dtype, tiled, on_input, flush=True)
    fm = moe.fused_moe
    x, w13, w2, tw, ids, kw = _args(moe, dev, T, E, K, H, I, dtype, tiled, skew)
    b13, b2 = torch.zeros(E, 2 * I, dtype=dtype, device=dev), torch.zeros(E, H, dtype=dtype, device=dev)
    so, eo, npp = fm.moe_align_block_size(ids, 256, E)

    def run(passes, b13=None, b2=None):
        out, ws = torch.full_like(x, float("nan")), None
        for p in passes:
            args = fm.launch_fused_experts(x, out, w13, w2, b13, b2, None, None, tw, so, eo, npp, 256, workspace=ws, passes=p,
                                           apply_router_weight_on_input=on_input, **kw)
            ws = args._keepalive[0]
        fm.fused_experts_status(args)
        return out

    want = run([7 | 8], b13, b2)
    assert bool(want.isfinite().all()) and float(want.float().abs().max()) > 0
    for passes in ([0], [7 | 8], [1, 2, 4], [7 | 32], [7 | 32]):
        assert torch.equal(run(passes), want), passes


def test_expired_wait_of_a_pair_is_nan_or_right(moe, dev):
    """A pair that gives up waiting leaves NaN in both its tiles: no element is anything but NaN or right."""
    x, w13, w2, tw, ids, kw = _args(moe, dev, 7600, 4, 2, 4096, 128, torch.bfloat16, False, 0.0)
    want = moe.fused_experts(x, w13, w2, None, None, tw, ids)
    torch.cuda.synchronize()
    before = moe.fused_moe.set_wait_limit(0)
    try:
        got = moe.fused_experts(x, w13, w2, None, None, tw, ids)
        torch.cuda.synchronize()
    finally:
        moe.fused_moe.set_wait_limit(before)
    assert bool((got.isnan() | (got == want)).all())
    assert torch.equal(moe.fused_experts(x, w13, w2, None, None, tw, ids), want)
