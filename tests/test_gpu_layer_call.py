"""The layer as one call into native code: the same results as its steps, and the kernels it picks by the sizes."""
import importlib
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
    """``fused_topk_experts`` against alignment and experts enqueued from Python with a block size of the caller's
    own, on rows that only the register-staged kernels take: equal up to the order of the sums."""
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


@pytest.mark.parametrize("E,H,I,K,T,layout", [(16, 4096, 1024, 2, 500, "plain"), (128, 256, 128, 2, 2048, "plain"),
                                              (128, 256, 128, 2, 2048, "tiled")])
def test_checked_hand_off_runs_the_kernels_of_the_call(moe, dev, monkeypatch, E, H, I, K, T, layout):
    """With the hand-off check on, the call is enqueued step by step: on the same kernels, with the same bits, where the
    rule by rows and tiles would take the other block size."""
    print(f"hand-off check E={E} H={H} I={I} T={T} {layout}", flush=True)
    g = torch.Generator(dev).manual_seed(T)
    normal = lambda *shape: torch.empty(shape, dtype=torch.bfloat16, device=dev).normal_(generator=g)
    x, logits, w13, w2 = normal(T, H), normal(T, E), normal(E, 2 * I, H) * 0.05, normal(E, H, I) * 0.05
    if layout == "tiled":
        w13, w2 = moe.ops.tile_expert_weights(w13, True), moe.ops.tile_expert_weights(w2, False)
    one = moe.fused_topk_experts(x, logits, w13, w2, K, True, weight_layout=layout)
    blocks, launch = [], moe.fused_moe.launch_fused_experts
    monkeypatch.setattr(moe.fused_moe, "launch_fused_experts",
                        lambda *a, **k: (blocks.append(a[12]), launch(*a, **k))[1])
    monkeypatch.setattr(moe.fused_moe, "_CHECK_HANDOFF", True)
    checked = moe.fused_topk_experts(x, logits, w13, w2, K, True, weight_layout=layout)
    assert blocks == [256 if E == 16 else 32]
    assert torch.equal(checked, one)


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


def _case(dev, T, E, K, H, I, dtype=torch.bfloat16, e4m3=False, tiled=False, activation="silu", bias=False, on_input=False,
          seed=1):
    """Arguments of ``fused_topk_experts``."""
    moe = importlib.import_module("layered-prefill_amd")
    g = torch.Generator().manual_seed(seed + T + H)
    draw = lambda *shape, std=1.0: (torch.randn(*shape, generator=g) * std).to(dtype).to(dev)
    x, logits = draw(T, H), draw(T, E)
    w13, w2 = draw(E, 2 * I, H, std=0.05), draw(E, H, I, std=0.05)
    kw = dict(activation=activation, apply_router_weight_on_input=on_input)
    if bias:
        kw.update(w1_bias=draw(E, 2 * I, std=0.1), w2_bias=draw(E, H, std=0.1))
    if e4m3:
        w13, kw["w1_scale"], w2, kw["w2_scale"] = moe.quantize_expert_weights(w13, w2)
    if tiled:
        w13 = moe.ops.tile_expert_weights(w13, True, activation == "swigluoai")
        w2, kw["weight_layout"] = moe.ops.tile_expert_weights(w2, False), "tiled"
    return x, logits, w13, w2, K, kw


_KERNELS = {
    "large tile": dict(T=700, E=8, K=2, H=256, I=128),
    "large tile, tiled weights": dict(T=700, E=8, K=2, H=256, I=128, dtype=torch.float16, tiled=True),
    "large tile, biased": dict(T=400, E=4, K=2, H=256, I=128, activation="swigluoai", bias=True),
    "large tile, e4m3": dict(T=900, E=16, K=4, H=256, I=128, e4m3=True),
    "streaming": dict(T=100, E=64, K=4, H=256, I=192),
    "streaming, tiled weights": dict(T=9, E=64, K=4, H=256, I=128, tiled=True),
    "streaming in place of the large tile": dict(T=200, E=16, K=4, H=512, I=256),
    "streaming, rows with a tail": dict(T=33, E=8, K=2, H=96, I=160, dtype=torch.float16),
    "streaming, e4m3": dict(T=60, E=16, K=4, H=256, I=128, e4m3=True),
    "streaming, e4m3 in place of the large tile": dict(T=200, E=16, K=4, H=256, I=128, e4m3=True),
    "streaming, biased": dict(T=150, E=32, K=4, H=256, I=128, activation="swigluoai", bias=True),
    "streaming, gelu, weight on the input": dict(T=40, E=8, K=1, H=128, I=64, activation="gelu", on_input=True),
    "element by element": dict(T=40, E=8, K=2, H=100, I=52),
    "fp32": dict(T=300, E=8, K=2, H=64, I=32, dtype=torch.float32),
}


@pytest.mark.parametrize("kernel", list(_KERNELS))
def test_one_call_has_the_bits_of_its_steps(moe, dev, monkeypatch, kernel):
    """The native entry against the same kernels enqueued from Python, with routing inside and outside the call, in
    place and on another stream; every size takes the native way."""
    print(kernel, flush=True)
    x, logits, w13, w2, K, kw = _case(dev, **_KERNELS[kernel])
    asked = []
    native = moe.fused_moe._layer_call
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: asked.append(native(*a)) or asked[-1])
    one = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    tw, ids, _ = moe.fused_topk(x, logits, K, True)
    rest = dict(kw)
    bias = rest.pop("w1_bias", None), rest.pop("w2_bias", None)
    routed = moe.fused_experts(x, w13, w2, *bias, tw, ids, **rest)
    inplace = x.clone()
    assert moe.fused_topk_experts(inplace, logits, w13, w2, K, True, inplace=True, **kw) is inplace
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    torch.cuda.current_stream().wait_stream(side)
    assert len(asked) == 4 and all(a is not None for a in asked)
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: None)
    steps = moe.fused_topk_experts(x, logits, w13, w2, K, True, **kw)
    assert bool(steps.isfinite().all()) and float(steps.float().abs().max()) > 0
    for got in (one, routed, inplace, other):
        assert torch.equal(got, steps)


def test_calls_from_several_threads_and_streams(moe, dev):
    """Each thread with a stream and a layer of its own, of different kernels; results as one after the other."""
    names = ["large tile", "streaming", "streaming, e4m3", "large tile, biased"]
    cases = [_case(dev, seed=7 + i, **_KERNELS[n]) for i, n in enumerate(names)]
    norm = moe.RMSNorm(256).bfloat16().to(dev)

    def run(c):
        x, logits, w13, w2, K, kw = c
        return moe.fused_topk_experts(norm(x), logits, w13, w2, K, True, **kw)

    want = [run(c) for c in cases]
    torch.cuda.synchronize()
    got, errors = [[] for _ in cases], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    got[i].append(run(cases[i]))
                torch.cuda.current_stream().synchronize()
        except Exception as e:   # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for w, results in zip(want, got):
        assert len(results) == 20 and all(torch.equal(w, r) for r in results)


def test_calls_that_are_not_plain_take_the_python_way(moe, dev, monkeypatch):
    """What the native entry answers with None has the result, or the error, of the Python path."""
    x, logits, w13, w2, K, kw = _case(dev, T=30, E=8, K=2, H=64, I=32)
    tw, ids, _ = moe.fused_topk(x, logits, K, True)
    want = moe.fused_topk_experts(x, logits, w13, w2, K, True)
    asked = []
    native = moe.fused_moe._layer_call
    monkeypatch.setattr(moe.fused_moe, "_layer_call", lambda *a: asked.append(native(*a)) or asked[-1])
    strided = torch.empty(30, 16, dtype=logits.dtype, device=dev)[:, ::2].copy_(logits)
    for call in (lambda: moe.fused_topk_experts(x, strided, w13, w2, K, True),
                 lambda: moe.fused_topk_experts(x, logits.double(), w13, w2, K, True),
                 lambda: moe.fused_experts(x, w13, w2, None, None, tw, ids.long()),
                 lambda: moe.fused_experts(x, w13, w2, None, None, tw.double(), ids),
                 lambda: moe.fused_experts(x, w13, w2, None, None, tw.t().contiguous().t(), ids)):
        asked.clear()
        out = call()
        assert asked[0] is None and torch.equal(out, want)
    with pytest.raises(AssertionError, match="must be contiguous"):
        moe.fused_topk_experts(x.t().contiguous().t(), logits, w13, w2, K, True)
    with pytest.raises(AssertionError, match="share a dtype"):
        moe.fused_topk_experts(x, logits, w13.half(), w2.half(), K, True)
    with pytest.raises(ValueError, match="Unsupported FusedMoe activation"):
        moe.fused_topk_experts(x, logits, w13, w2, K, True, activation="relu")
    with pytest.raises(RuntimeError, match="exceeds num_experts"):
        moe.fused_topk_experts(x, logits, w13, w2, 9, True)
    assert moe.fused_topk_experts(x[:0], logits[:0], w13, w2, K, True).shape == (0, 64)
    # e4m3 codes as bytes, and more tokens than a chunk
    x8, logits8, q13, q2, _, kw8 = _case(dev, T=30, E=8, K=2, H=64, I=32, e4m3=True)
    assert torch.equal(moe.fused_topk_experts(x8, logits8, q13.view(torch.uint8), q2.view(torch.uint8), K, True, **kw8),
                       moe.fused_topk_experts(x8, logits8, q13, q2, K, True, **kw8))
    xl, logitsl, v13, v2, _, _ = _case(dev, T=65536 + 30, E=2, K=1, H=32, I=16)
    asked.clear()
    long = moe.fused_topk_experts(xl, logitsl, v13, v2, 1, True)
    assert asked[0] is None
    assert torch.equal(long[:65536], moe.fused_topk_experts(xl[:65536], logitsl[:65536], v13, v2, 1, True))
    assert torch.equal(long[65536:], moe.fused_topk_experts(xl[65536:], logitsl[65536:], v13, v2, 1, True))
