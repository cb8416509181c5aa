"""Results of the native host calls are made past the dispatcher only where it would make the same ones."""
import pytest
import torch
from torch.profiler import ProfilerActivity, profile
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.empties = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.empties += func in (torch.ops.aten.empty.memory_format,)
        return func(*args, **(kwargs or {}))


def _profiled(run):
    """What it returns, and how many tensors the dispatcher was asked for."""
    with profile(activities=[ProfilerActivity.CPU]) as p:
        got = run()
    return got, sum(e.name == "aten::empty" for e in p.events())


@pytest.mark.parametrize("form", ["plain", "mode", "inference", "deterministic"])
def test_results_are_what_empty_makes(moe, dev, form):
    print(form, flush=True)
    g = torch.Generator(dev).manual_seed(5)
    x = torch.randn(20, 256, generator=g, device=dev).bfloat16()
    logits = torch.randn(20, 32, generator=g, device=dev).bfloat16()
    norm = moe.RMSNorm(256).to(device=dev, dtype=torch.bfloat16)
    host = moe._lib.host()
    run = lambda: [host.rms_norm(x, None, norm.weight.data, norm.eps), *host.topk(logits, 4, True)]
    want, seen = run(), None
    if form == "mode":
        with _Seen() as seen:
            got = run()
    elif form == "inference":
        with torch.inference_mode():
            got, through = _profiled(run)
    elif form == "deterministic":
        before = torch.are_deterministic_algorithms_enabled(), torch.is_deterministic_algorithms_warn_only_enabled()
        torch.use_deterministic_algorithms(True)
        try:
            got, through = _profiled(run)
        finally:
            torch.use_deterministic_algorithms(before[0], warn_only=before[1])
    else:
        got, through = _profiled(run)
    if seen is not None:
        through = seen.empties
    assert through == (4 if form in ("mode", "deterministic") else 0)
    for a, b in zip(got, want):
        assert torch.equal(a, b) and a.device == x.device and a.is_contiguous() and not a.requires_grad
        assert a.is_inference() == (form == "inference") and a.dtype == b.dtype
        assert a.untyped_storage().nbytes() == a.numel() * a.element_size()
