"""Alignment over several workgroups: the sizes at which a workgroup, an instance or the way it counts changes, against
the oracle, with and without blocks of 256 and on skewed, repeated and invalid ids."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ids(numel, E, kind):
    g = torch.Generator().manual_seed(numel + E)
    if kind == "one":
        return torch.full((numel,), E - 1, dtype=torch.int32)
    ids = (torch.rand(numel, generator=g) ** 4 * E).int().clamp(max=E - 1)
    if kind == "holes":   # ids of no expert are left out
        ids[torch.rand(numel, generator=g) < 0.1] = E
        ids[torch.rand(numel, generator=g) < 0.1] = -1
    return ids


@pytest.mark.parametrize("numel", [1023, 1024, 1025, 2049, 8191, 8192, 8193, 16384, 16385, 17000, 67585])
@pytest.mark.parametrize("E,block,kind", [(128, 256, "skewed"), (256, 32, "skewed"), (1, 64, "skewed"), (100, 16, "holes"),
                                          (5, 256, "one")])
def test_alignment_at_the_seams(moe, oracle, dev, numel, E, block, kind):
    ids = _ids(numel, E, kind)
    got = moe.moe_align_block_size(ids.view(-1, 1).to(dev), block, E)
    if kind == "holes":   # by the definition: the oracle takes ids of experts only
        want = torch.full_like(got[0].cpu(), numel)
        experts, at = [], 0
        for e in range(E):
            mine = (ids == e).nonzero().flatten().int()
            want[at:at + len(mine)] = mine
            blocks = -(-len(mine) // block)
            experts += [e] * blocks
            at += blocks * block
        assert got[2].item() == at and torch.equal(got[0].cpu(), want)
        assert got[1].cpu()[:len(experts)].tolist() == experts
        return
    want = oracle.moe_align_block_size(ids.view(-1, 1), block, E)
    assert all(torch.equal(a.cpu(), b) for a, b in zip(got, want))


@pytest.mark.parametrize("numel", [1030, 6000, 16384, 20000, 100000])
def test_plan_of_many_workgroups_is_that_of_the_ids(moe, dev, numel):
    """The expert passes on a plan that the alignment left, and on the one that they make from the aligned ids."""
    E, K, H, I = 64, 2, 256, 128
    T = numel // K
    g = torch.Generator(dev).manual_seed(numel)
    x = torch.empty(T, H, dtype=torch.bfloat16, device=dev).normal_(0, 1, generator=g)
    w13 = torch.empty(E, 2 * I, H, dtype=torch.bfloat16, device=dev).normal_(0, 0.05, generator=g)
    w2 = torch.empty(E, H, I, dtype=torch.bfloat16, device=dev).normal_(0, 0.05, generator=g)
    ids = _ids(T * K, E, "skewed").view(T, K).to(dev)
    tw = torch.rand(T, K, device=dev)
    out = moe.fused_experts(x, w13, w2, None, None, tw, ids)
    want = torch.zeros(T, H, device=dev)
    for k in range(K):   # one expert at a time, fp32 from the same bf16 inputs
        for e in range(E):
            rows = (ids[:, k] == e).nonzero().flatten()
            if len(rows):
                gu = x[rows].float() @ w13[e].float().t()
                h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]).bfloat16().float()
                want[rows] += tw[rows, k, None] * (h @ w2[e].float().t())
    # roundings of the intermediate, of each term and of the sum: 3 of 2^-9 relative, sums of 128 and 256 products in fp32
    err = (out.float() - want).norm() / want.norm()
    assert err < 3 * 2 ** -8
