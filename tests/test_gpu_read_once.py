"""Kernels that read a large buffer once and past the caches: sizes beyond those of the other tests, where a launch has
more workgroups than fit the card, and right behind the kernel that wrote the buffer."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,H,dtype", [(4099, 8, 2048, torch.bfloat16), (16385, 4, 520, torch.float16),
                                         (9001, 3, 1032, torch.bfloat16), (2100, 8, 1028, torch.float32),
                                         # on both sides of the lines from which the terms are read past the caches
                                         (7680, 8, 1024, torch.bfloat16), (7681, 8, 1024, torch.bfloat16),
                                         (15500, 4, 1024, torch.float16), (9001, 7, 1024, torch.bfloat16),
                                         (12000, 8, 1000, torch.float16), (17000, 6, 1000, torch.bfloat16),
                                         (12500, 4, 1000, torch.float32), (13100, 3, 1024, torch.float32)])
def test_combine_of_many_rows(moe, dev, T, K, H, dtype):
    g = torch.Generator(dev).manual_seed(T)
    rows = torch.empty(T, K, H, dtype=dtype, device=dev)
    out = torch.full((T, H), float("nan"), dtype=dtype, device=dev)
    for _ in range(3):  # (the rows change under it: nothing of the last pass may be read again)
        rows.normal_(0, 1, generator=g)
        moe.ops.moe_sum(rows, out)
        want = torch.zeros(T, H, dtype=torch.float32, device=dev)
        for k in range(K):
            want += rows[:, k].float()
        assert torch.equal(out, want.to(dtype))
