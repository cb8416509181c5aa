"""exp of the activations at and beyond the ends of its range, in wavefronts all inside it, all outside and mixed: bits of the
oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_silu_at_the_ends_of_the_range(moe, oracle, dev, dtype):
    g = torch.Generator().manual_seed(11)
    d = 1024
    ends = torch.tensor([0.0, -0.0, 85.99, 86.0, 86.01, 87.3, 88.0, 88.01, 103.9, 104.0, 104.1, 1e30, float("inf"), float("nan"), 1e-40])
    ends = torch.cat([ends, -ends])
    gates = [torch.randn(d, generator=g), torch.full((d,), 90.0), torch.full((d,), -95.0), torch.linspace(-110.0, 110.0, d)]
    gates += [torch.linspace(80.0, 110.0, d), torch.linspace(-110.0, -80.0, d), ends.repeat(d)[:d]]
    for i, v in enumerate(ends.tolist()):   # one lane of a row
        row = torch.randn(d, generator=g)
        row[(37 * i) % d] = v
        gates.append(row)
    x = torch.cat([torch.stack(gates), torch.randn(len(gates), d, generator=g)], dim=1).to(getattr(torch, dtype))
    out = torch.empty(len(gates), d, dtype=x.dtype, device=dev)
    moe.ops.silu_and_mul(out, x.to(dev))
    got, want = out.cpu(), oracle.silu_and_mul(x)
    assert torch.equal(got.isnan(), want.isnan())
    bits = torch.int32 if dtype == "float32" else torch.int16
    ok = ~want.isnan()
    assert torch.equal(got[ok].view(bits), want[ok].view(bits))
