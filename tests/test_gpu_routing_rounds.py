"""Rounds of the router over sorted lanes: order of equals inside a lane and across lanes, all columns of a row taken,
rows of NaN beside rows of numbers in a wavefront, more winners than a row has lanes.  Bits of the oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("values", [1, 2, 7, 1000])
def test_equal_values_leave_in_column_order(moe, oracle, dev, E, values):
    print(E, values, flush=True)
    g = torch.Generator().manual_seed(E + values)
    T = 67
    logits = torch.randint(0, values, (T, E), generator=g).float() * 0.25
    logits[3, : E // 2] = float("-inf")       # probabilities that are exactly zero: the last to leave, in column order
    for K in sorted({1, 3, E // 4, E // 2, E}):
        for renormalize in (False, True):
            w, ids, tei = moe.fused_topk(torch.zeros(T, 8, device=dev), logits.to(dev), K, renormalize)
            ow, oids, otei = oracle.fused_topk(torch.zeros(T, 8), logits, K, renormalize)
            assert torch.equal(ids.cpu(), oids) and torch.equal(tei.cpu(), otei)
            assert torch.equal(w.cpu().view(torch.int32), ow.view(torch.int32))


@pytest.mark.parametrize("E", [8, 32, 128])
def test_rows_of_nan_do_not_change_their_neighbours(moe, oracle, dev, E):
    g = torch.Generator().manual_seed(E)
    T, K = 40, 4
    logits = torch.randn(T, E, generator=g)
    bad = torch.zeros(T, dtype=torch.bool)
    bad[torch.arange(1, T, 5)] = True
    broken = logits.clone()
    broken[bad, E // 3] = float("nan")
    w, ids, _ = moe.fused_topk(torch.zeros(T, 8, device=dev), broken.to(dev), K, True)
    ow, oids, _ = oracle.fused_topk(torch.zeros(T, 8), logits, K, True)
    assert torch.equal(ids.cpu()[~bad], oids[~bad])
    assert torch.equal(w.cpu()[~bad].view(torch.int32), ow[~bad].view(torch.int32))
    assert bool(w.cpu()[bad].isnan().all()) and not ids.cpu()[bad].any()


@pytest.mark.parametrize("E,lanes", [(1, 1), (2, 1), (4, 1), (8, 2), (16, 4), (32, 8), (64, 16), (128, 32), (256, 32)])
@pytest.mark.parametrize("T", [1, 67])
def test_more_winners_than_a_row_has_lanes(moe, oracle, dev, E, lanes, T):
    print(E, T, flush=True)
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(E + T))
    for K in sorted(k for k in {1, lanes - 1, lanes, lanes + 1, 2 * lanes - 1, 2 * lanes, 3 * lanes + 1, E - 1, E} if 1 <= k <= E):
        for renormalize in (False, True):
            w, ids, tei = moe.fused_topk(torch.zeros(T, 8, device=dev), logits.to(dev), K, renormalize)
            ow, oids, otei = oracle.fused_topk(torch.zeros(T, 8), logits, K, renormalize)
            assert torch.equal(ids.cpu(), oids) and torch.equal(tei.cpu(), otei)
            assert torch.equal(w.cpu().view(torch.int32), ow.view(torch.int32))


@pytest.mark.parametrize("T,E,K", [(1, 16, 6), (9, 8, 8), (40, 16, 9), (60, 32, 17), (700, 16, 6)])
@pytest.mark.parametrize("e4m3", [False, True])
def test_more_winners_than_lanes_inside_a_layer(moe, dev, monkeypatch, T, E, K, e4m3):
    """Routing with alignment, and beside the quantisation: the bits of the steps, whose routing stands alone."""
    print(T, E, K, e4m3, flush=True)
    g = torch.Generator(dev).manual_seed(T)
    draw = lambda *shape, std=1.0: torch.empty(shape, device=dev).normal_(0.0, std, generator=g).bfloat16()
    x, logits, w13, w2, kw = draw(T, 512), draw(T, E), draw(E, 768, 512, std=0.05), draw(E, 512, 384, std=0.05), {}
    if e4m3:
        w13, kw["w1_scale"], w2, kw["w2_scale"] = moe.quantize_expert_weights(w13, w2)
    run = lambda renormalize: moe.fused_topk_experts(x, logits, w13, w2, K, renormalize, **kw)
    got = [run(True), run(False)]
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    for a, renormalize in zip(got, (True, False)):
        want = run(renormalize)
        assert bool(want.isfinite().all()) and float(want.float().abs().max()) > 0
        assert torch.equal(a, want)
