"""Rounds of the router over sorted lanes: order of equals inside a lane and across lanes, all columns of a row taken,
rows of NaN beside rows of numbers in a wavefront.  Bits of the oracle."""
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
