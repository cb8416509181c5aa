"""The layer as one call into native code: the same results as its steps, and the kernels it picks by the sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,K", [(1, 1, 1), (3, 60, 4), (67, 128, 8), (33, 256, 8), (129, 300, 6), (5, 130, 130)])
def test_topk_of_16bit_logits_is_topk_of_their_float(moe, dev, dtype, T, E, K):
    print(f"topk {dtype} T={T} E={E} K={K}", flush=True)
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(T + E)).to(dtype).to(dev)
    x = torch.empty(T, 8, dtype=dtype, device=dev)
    for a, b in zip(moe.fused_topk(x, logits, K, True), moe.fused_topk(x, logits.float(), K, True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,activation,on_input", [(1, "silu", False), (40, "gelu", True), (700, "swigluoai", False)])
def test_one_call_is_its_steps(moe, dev, monkeypatch, T, activation, on_input):
    """``fused_topk_experts`` against alignment and experts enqueued from Python (what a block size of the
    caller's own takes), on sizes whose kernels are the same ones."""
    print(f"layer T={T} {activation}", flush=True)
    E, K, H, I = 8, 2, 136, 72
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, H, generator=g).bfloat16().to(dev)
    w13 = (torch.randn(E, 2 * I, H, generator=g) * 0.05).bfloat16().to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * 0.05).bfloat16().to(dev)
    logits = torch.randn(T, E, generator=g).bfloat16().to(dev)
    kw = dict(activation=activation, apply_router_weight_on_input=on_input)
    one = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    own = moe.fused_moe.try_get_optimal_moe_config
    monkeypatch.setattr(moe.fused_moe, "try_get_optimal_moe_config", lambda *a, **k: own(*a, **k))
    steps = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    assert (one.float() - steps.float()).norm() <= 2e-3 * steps.float().norm()
