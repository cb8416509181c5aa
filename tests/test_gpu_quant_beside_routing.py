"""The e4m3 codes of x made in the routing's launch: the bits of the steps enqueued one by one, at the edges of the instances."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,H,I,dtype,logits", [
    (1, 32, 4, 64, 64, "bfloat16", None),        # the router's launch, as wherever the gate-up pass aligns
    (16, 128, 8, 2048, 128, "float16", None),    # the widest rows of its narrower instance
    (17, 128, 8, 2048, 64, "bfloat16", None),
    # beside routing and alignment in one launch: up to 2048 logits, rows that are no whole 32 bytes
    (1, 32, 4, 2000, 64, "bfloat16", None),      # one row, up to 2048 columns
    (16, 128, 8, 2000, 128, "float16", None),    # the most logits of it, a whole workgroup of rows
    (17, 64, 2, 2064, 64, "bfloat16", None),     # rows of more than 2048 columns, a second workgroup of them
    (8, 256, 8, 4080, 64, "float16", None),      # the widest rows
    (33, 64, 2, 2000, 64, "bfloat16", None),     # one row too many: the router's launch
    (33, 16, 2, 4096, 64, "float16", None),
    (130, 256, 4, 2064, 64, "bfloat16", None),
    (700, 8, 2, 256, 128, "bfloat16", None),     # experts without an instance
    (40, 64, 2, 4112, 64, "bfloat16", None),     # rows too long
    (40, 64, 2, 256, 64, "bfloat16", "float32"), # logits of another type
])
def test_codes_beside_the_routing_have_the_bits_of_the_steps(moe, dev, monkeypatch, T, E, K, H, I, dtype, logits):
    print(T, E, K, H, I, dtype, logits, flush=True)
    g = torch.Generator().manual_seed(T + E + H)
    dt = getattr(torch, dtype)
    x = (torch.randn(T, H, generator=g) * torch.rand(T, 1, generator=g) * 8).to(dt).to(dev)
    if T > 1:
        x[T // 2] = 0   # a row whose scale is 1
    lg = torch.randn(T, E, generator=g).to(getattr(torch, logits or dtype)).to(dev)
    w13 = (torch.randn(E, 2 * I, H, generator=g) * 0.05).to(dt).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.05).to(dt).to(dev)
    q13, s13, q2, s2 = moe.quantize_expert_weights(w13, w2)
    kw = dict(w1_scale=s13, w2_scale=s2)
    one = moe.fused_topk_experts(x, lg, q13, q2, K, True, **kw)
    inplace = x.clone()
    moe.fused_topk_experts(inplace, lg, q13, q2, K, True, inplace=True, **kw)
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = moe.fused_topk_experts(x, lg, q13, q2, K, True, **kw)
    assert bool(steps.isfinite().all()) and float(steps.float().abs().max()) > 0
    assert torch.equal(one, steps) and torch.equal(inplace, steps)
