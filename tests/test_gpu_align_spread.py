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


@pytest.mark.parametrize("numel", [1023, 1024, 1025, 2049, 8191, 8192, 8193, 16384, 16385, 17000, 67585, 262144])
@pytest.mark.parametrize("E,block,kind", [(128, 256, "skewed"), (256, 32, "skewed"), (1, 64, "skewed"), (100, 16, "holes"),
                                          (5, 256, "one"), (3, 1, "skewed"), (2, 32, "holes"), (4, 256, "holes"),
                                          (1, 256, "one")])
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


@pytest.mark.parametrize("E,K", [(64, 2), (200, 1), (3, 1)])
@pytest.mark.parametrize("numel", [1030, 6000, 8194, 12000, 16384, 20000, 100000])
def test_plan_of_many_workgroups_is_that_of_the_ids(moe, dev, numel, E, K):
    """The expert passes on a plan that the alignment left in a workspace of other contents, and on the one that they make
    from the aligned ids: the same ranges, the same bits."""
    print(numel, E, K, flush=True)
    fm = moe.fused_moe
    H, I, T = 256, 128, numel // K
    g = torch.Generator(dev).manual_seed(numel)
    x = torch.empty(T, H, dtype=torch.bfloat16, device=dev).normal_(0, 1, generator=g)
    w13 = torch.empty(E, 2 * I, H, dtype=torch.bfloat16, device=dev).normal_(0, 0.05, generator=g)
    w2 = torch.empty(E, H, I, dtype=torch.bfloat16, device=dev).normal_(0, 0.05, generator=g)
    ids = _ids(T * K, E, "skewed").view(T, K).to(dev)
    tw = torch.rand(T, K, device=dev)
    code = moe._lib.DTYPE_CODE[torch.bfloat16]
    size = fm.fused_experts_workspace_bytes(T, H, I, E, K, 256, torch.bfloat16)
    out, ranges = [], []
    for planned in (True, False):
        ws = torch.full((size,), 0x5a, dtype=torch.uint8, device=dev)
        plan = fm._plan_in_workspace(ws, T, H, I, E, K, 256, code, code, T * K)
        assert plan is not None
        so, eo, npp = fm._align_block_size(ids, 256, E, plan if planned else None)
        out.append(torch.full_like(x, float("nan")))
        args = fm.launch_fused_experts(x, out[-1], w13, w2, None, None, None, None, tw, so, eo, npp, 256, workspace=ws,
                                       passes=16 if planned else 0)
        fm.fused_experts_status(args)
        at = plan[0] - ws.data_ptr()
        ranges.append(ws[at:at + 36].clone().view(torch.int32).tolist())
    assert ranges[0] == ranges[1] and ranges[0][0] == 0 and ranges[0][8] == npp.item() // 256
    assert bool(out[1].isfinite().all()) and torch.equal(out[0], out[1])
    want = torch.zeros(T, H, device=dev)
    for k in range(K):   # one expert at a time, fp32 from the same bf16 inputs
        for e in range(E):
            rows = (ids[:, k] == e).nonzero().flatten()
            if len(rows):
                gu = x[rows].float() @ w13[e].float().t()
                h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]).bfloat16().float()
                want[rows] += tw[rows, k, None] * (h @ w2[e].float().t())
    # roundings of the intermediate, of each term and of the sum: 3 of 2^-9 relative, sums of 128 and 256 products in fp32
    err = (out[0].float() - want).norm() / want.norm()
    assert err < 3 * 2 ** -8


@pytest.mark.parametrize("cap", [2 ** 31 - 1 - 2 ** 20, 2 ** 31 - 2 ** 20, 2 ** 31 - 1])
@pytest.mark.parametrize("numel", [300, 1500, 20000])
def test_longest_outputs(moe, oracle, dev, numel, cap):
    """Output buffers up to the largest length there is, on both sides of the line behind which slots are counted in 64 bits:
    all of them is written, and nothing in front of it."""
    print(numel, cap, flush=True)
    E, block, guard = 8, 32, 1024
    ids = _ids(numel, E, "skewed")
    want = oracle.moe_align_block_size(ids.view(-1, 1), block, E)
    whole = torch.full((guard + cap,), -7, dtype=torch.int32, device=dev)   # 8.6 GB
    experts = torch.full((want[1].numel() + 100,), -7, dtype=torch.int32, device=dev)
    total = torch.empty(1, dtype=torch.int32, device=dev)
    slots = whole[guard:]
    moe.ops.moe_align_block_size(ids.to(dev), E, block, slots, experts, total)
    need = want[0].numel()
    assert torch.equal(slots[:need].cpu(), want[0]) and torch.equal(total.cpu(), want[2])
    assert torch.equal(experts[:want[1].numel()].cpu(), want[1]) and not bool(experts[want[1].numel():].any())
    for at in range(need, cap, 1 << 28):
        assert bool((slots[at:at + (1 << 28)] == numel).all())
    assert bool((whole[:guard] == -7).all())
    del whole, slots
    torch.cuda.empty_cache()
