"""The layer as one call into native code: the same results as its steps, and the kernels it picks by the sizes."""
import sys
import threading

import numpy as np
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("E,K", [(1, 1), (2, 1), (4, 2), (8, 2), (32, 4), (128, 8), (256, 8), (60, 4), (1100, 2)])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_logits_need_the_alignment_of_an_element_only(moe, dev, dtype, E, K, offset):
    print(f"logits {dtype} E={E} offset={offset}", flush=True)
    T, H, I = 9, 32, 32
    g = torch.Generator().manual_seed(E + offset)
    aligned = torch.randn(T, E, generator=g).to(dtype).to(dev)
    buf = torch.full((T * E + 8,), 50.0, dtype=dtype, device=dev)
    logits = buf[offset:offset + T * E].view(T, E).copy_(aligned)
    assert logits.is_contiguous() and logits.data_ptr() % 16 == offset * logits.element_size()
    x = torch.randn(T, H, generator=g).bfloat16().to(dev)
    for a, b in zip(moe.fused_topk(x, logits, K, True), moe.fused_topk(x, aligned, K, True)):
        assert torch.equal(a, b)
    if E <= 256:
        w13 = torch.randn(E, 2 * I, H, generator=g).bfloat16().to(dev)
        w2 = torch.randn(E, H, I, generator=g).bfloat16().to(dev)
        assert torch.equal(moe.fused_topk_experts(x, logits, w13, w2, K, True),
                           moe.fused_topk_experts(x, aligned, w13, w2, K, True))


@pytest.mark.parametrize("shape", [(4,), (4, 2, 8)])
def test_routing_refuses_hidden_states_that_are_no_matrix(moe, dev, shape):
    x = torch.zeros(shape, dtype=torch.bfloat16, device=dev)
    logits = torch.zeros(4, 8, device=dev)
    with pytest.raises(ValueError):
        moe.fused_topk(x, logits, 2, True)
    w = torch.zeros(8, 16, 8, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        moe.fused_topk_experts(x, logits, w, w[:, :, :8], 2, True)


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


def test_arguments_are_converted_or_refused_as_python_does(moe, dev):
    """What is no plain int, bool or float takes the Python path: what converts, converts; what does not is that
    path's error, in front of any launch."""
    g = torch.Generator().manual_seed(3)
    x = torch.randn(5, 32, generator=g).bfloat16().to(dev)
    logits = torch.randn(5, 8, generator=g).bfloat16().to(dev)
    w13 = (torch.randn(8, 64, 32, generator=g) * 0.1).bfloat16().to(dev)
    w2 = (torch.randn(8, 32, 32, generator=g) * 0.1).bfloat16().to(dev)
    gate = torch.randn(32, 64, generator=g).bfloat16().to(dev)
    many = torch.randn(2048, 64, generator=g).bfloat16().to(dev)
    plain = moe.fused_topk(x, logits, 2, True)
    for topk, renormalize in ((np.int64(2), True), (2, np.bool_(True)), (2, 1)):
        assert all(torch.equal(a, b) for a, b in zip(moe.fused_topk(x, logits, topk, renormalize), plain))
    for topk in (2.0, "2", None):
        with pytest.raises(TypeError):
            moe.fused_topk(x, logits, topk, True)
        with pytest.raises(TypeError):
            moe.fused_topk_experts(x, logits, w13, w2, topk, True)
        with pytest.raises(TypeError):
            moe.fused_gate_topk(many, gate, topk, True)
    with pytest.raises((RuntimeError, OverflowError, TypeError)):
        moe.fused_topk(x, logits, 1 << 70, True)
    for renormalize in (None, [1]):
        with pytest.raises(TypeError):
            moe.fused_topk(x, logits, 2, renormalize)
    out = moe.fused_topk_experts(x, logits, w13, w2, 2, True)
    for kw in (dict(apply_router_weight_on_input=np.bool_(False)), dict(inplace=0), dict(inplace=None)):
        assert torch.equal(moe.fused_topk_experts(x, logits, w13, w2, np.int64(2), np.bool_(True), **kw), out)

    norm, res = moe.RMSNorm(32, eps="1e-6").bfloat16().to(dev), x.clone()
    want, want_res = moe.RMSNorm(32).bfloat16().to(dev)(x, x.clone())
    got, _ = norm(x, res)
    assert torch.equal(got, want) and torch.equal(res, want_res)
    norm.eps, res = None, x.clone()
    with pytest.raises(TypeError):
        norm(x, res)
    assert torch.equal(res, x)


@pytest.mark.parametrize("call", ["layer", "topk", "norm", "gate"])
def test_other_python_threads_run_during_a_call(moe, dev, call):
    """With a switch interval of minutes a thread gets the interpreter only when the other gives it up: the calls
    have to.  (A release of microseconds may pass before the waiting thread is awake, hence the many
    calls; their results are kept, because torch gives the interpreter up where it frees a tensor.)"""
    x = torch.zeros(2048, 64, dtype=torch.bfloat16, device=dev)
    logits = torch.zeros(2048, 32, dtype=torch.bfloat16, device=dev)
    w13, w2 = (torch.zeros(32, n, k, dtype=torch.bfloat16, device=dev) for n, k in ((64, 64), (64, 32)))
    norm = moe.RMSNorm(64).bfloat16().to(dev)
    run = {"layer": lambda: moe.fused_topk_experts(x[:1], logits[:1], w13, w2, 2, True),
           "topk": lambda: moe.fused_topk(x, logits, 2, True),
           "norm": lambda: norm(x),
           "gate": lambda: moe.fused_gate_topk(x, x[:32], 2, True)}[call]
    native = {"layer": "layer", "topk": "topk", "norm": "rms_norm", "gate": "gate_topk"}[call]
    args = []
    host = moe._lib.host()

    class Recorder:   # the arguments of the native call, so that the loop below makes nothing but that call
        def __getattr__(self, name):
            def f(*a):
                args.append((name, a))
                return getattr(host, name)(*a)
            return f

    own = moe._lib.host
    moe._lib.host = lambda: Recorder()
    try:
        run()
    finally:
        moe._lib.host = own
    a = next(a for name, a in args if name == native)
    enter = getattr(host, native)
    assert enter(*a) is not None
    torch.cuda.synchronize()
    ran, go = [], threading.Event()

    def other():
        go.wait()
        ran.append(1)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    thread.start()
    sys.setswitchinterval(600.0)
    try:
        go.set()
        results = []
        for _ in range(10000):
            results.append(enter(*a))
            if ran:
                break
    finally:
        sys.setswitchinterval(interval)
    assert ran
    thread.join()
