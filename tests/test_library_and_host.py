"""CPU-only checks: the C-ABI library loads and exports what include/*.h
declares, argument validation rejects bad calls before touching a GPU, the
host-side mirror of the reference interface behaves, and the workloads are
reproducible.  No kernel is launched here."""
import ctypes
import inspect
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "moe_gfx950.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(moe_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = _declared_functions()
    for must in ("moe_topk_softmax", "moe_align_block_size", "moe_silu_and_mul", "moe_fused_experts",
                 "moe_sum", "moe_last_error", "moe_fused_experts_workspace_bytes"):
        assert must in names


def test_library_exports_every_declared_symbol(moe):
    lib = ctypes.CDLL(moe._lib.LIB_PATH)
    for name in _declared_functions():
        assert hasattr(lib, name), f"{name} declared in include/moe_gfx950.h but not exported"
    assert set(_declared_functions()) == set(moe._lib.EXPORTS)
    assert moe._lib.lib().moe_abi_version() == 2


def test_struct_layout_matches_header(moe):
    # field order of the ctypes mirror follows the C struct
    text = open(os.path.join(ROOT, "include", "moe_gfx950.h")).read()
    body = text[text.index("typedef struct MoeFusedExpertsArgs {"):text.index("} MoeFusedExpertsArgs;")]
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    c_fields = []
    for decl in body.split(";"):
        decl = decl.replace("typedef struct MoeFusedExpertsArgs {", "").strip()
        if not decl:
            continue
        names = decl.split(",")
        first = names[0].split()[-1].lstrip("*")
        c_fields.append(first)
        c_fields.extend(n.strip().lstrip("*") for n in names[1:])
    assert c_fields == [f[0] for f in moe._lib.MoeFusedExpertsArgs._fields_]


def test_argument_validation_without_gpu(moe):
    L = moe._lib.lib()
    assert L.moe_topk_softmax(None, None, None, None, 4, 8, 9, 0, None) == -1
    assert b"exceeds num_experts" in L.moe_last_error()
    assert L.moe_topk_softmax(None, None, None, None, 4, 20000, 2, 0, None) == -2
    assert L.moe_align_block_size(None, 0, 10, 2000, 16, None, 0, None, 0, None, None, 0, None) == -2
    assert L.moe_align_block_size(None, 9, 10, 8, 16, None, 0, None, 0, None, None, 0, None) == -1
    assert L.moe_silu_and_mul(None, None, 4, 0, 2, None) == -1
    assert L.moe_fused_experts(None) == -1
    assert L.moe_topk_softmax(None, None, None, None, 0, 8, 2, 0, None) == 0  # empty batch is a no-op
    assert L.moe_align_workspace_bytes(2048, 128) == 0
    assert L.moe_align_workspace_bytes(67584, 128) >= (132 * 128 + 129) * 4
    want = 0
    for rows, cols in ((67584 + 128 * 127, 768), (67584, 2048)):
        want += -(-rows * cols * 2 // 256) * 256
    # + one counter per 256-slot block (one-launch form of the large-tile passes) + XCD range table
    counters = -(-(-(-(67584 + 128 * 127) // 256) * 4) // 256) * 256
    assert L.moe_fused_experts_workspace_bytes(8448, 2048, 768, 128, 8, 128, 2, 2) == want + counters + 256
    # act dtype code 2 = bf16: streaming blocks, then the large tile from 16 rows per expert on
    for m, bm in ((64, 32), (192, 32), (256, 256), (512, 256), (768, 256), (8448, 256)):
        assert L.moe_preferred_block_size(m, 128, 8, 2, 2) == bm
    # e4m3 weights (code 3) quantise the intermediate between the passes: from 32 rows per expert on
    for m, bm in ((256, 32), (384, 32), (512, 256), (8448, 256)):
        assert L.moe_preferred_block_size(m, 128, 8, 2, 3) == bm
    # fp32 (code 0) has no large-tile kernel: the M tile follows the load
    for m, bm in ((256, 32), (768, 64), (2048, 128), (8448, 256)):
        assert L.moe_preferred_block_size(m, 128, 8, 0, 0) == bm


def test_ops_refuse_cpu_tensors(moe):
    ids = torch.zeros(4, 2, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="no CPU path"):
        moe.moe_align_block_size(ids, 16, 8)
    x = torch.zeros(4, 8)
    with pytest.raises(RuntimeError, match="no CPU path"):
        moe.fused_topk(x, torch.zeros(4, 8), 2, True)
    with pytest.raises(RuntimeError, match="no CPU path"):
        moe.ops.silu_and_mul(torch.zeros(4, 4), x)


def test_signatures_match_the_reference_interface(moe):
    # nanovllm/layers/for_moe/fused_moe.py:17-19,393-398,422-442
    assert list(inspect.signature(moe.moe_align_block_size).parameters) == ["topk_ids", "block_size", "num_experts"]
    assert list(inspect.signature(moe.fused_topk).parameters) == ["hidden_states", "gating_output", "topk", "renormalize"]
    fe = inspect.signature(moe.fused_experts).parameters
    # the reference's parameters, in its order; what this build adds comes after them, with a default
    assert list(fe)[:21] == ["hidden_states", "w1", "w2", "w1_bias", "w2_bias", "topk_weights", "topk_ids", "inplace",
                             "activation", "apply_router_weight_on_input", "per_channel_quant", "global_num_experts",
                             "expert_map", "w1_scale", "w2_scale", "w1_zp", "w2_zp", "a1_scale", "a2_scale",
                             "block_shape", "allow_deep_gemm"]
    assert list(fe)[21:] == ["weight_layout"] and fe["weight_layout"].default == "plain"
    assert fe["inplace"].default is False and fe["activation"].default == "silu"
    # csrc/ops.cpp:29-31,46-60
    assert list(inspect.signature(moe.ops.topk_softmax).parameters)[:4] == [
        "topk_weights", "topk_indices", "token_expert_indices", "gating_output"]
    assert list(inspect.signature(moe.ops.moe_align_block_size).parameters) == [
        "topk_ids", "num_experts", "block_size", "sorted_token_ids", "experts_ids", "num_tokens_post_pad"]
    assert list(inspect.signature(moe.ops.silu_and_mul).parameters) == ["out", "input"]


def test_fused_moe_module_parameters(moe):
    # nanovllm/layers/fused_moe.py:119-157: w13 [E, 2I, H], w2 [E, H, I] (+ biases)
    layer = moe.FusedMoE(8, 2, 256, 128, params_dtype=torch.bfloat16, has_bias=True)
    assert tuple(layer.w13_weight.shape) == (8, 256, 256) and layer.w13_weight.dtype == torch.bfloat16
    assert tuple(layer.w2_weight.shape) == (8, 256, 128)
    assert tuple(layer.w13_bias.shape) == (8, 256) and tuple(layer.w2_bias.shape) == (8, 256)
    assert not layer.w13_weight.requires_grad
    assert layer.tp_size == 1 and layer.tp_rank == 0 and layer.renormalize and layer.activation == "silu"
    with pytest.raises(ValueError, match="Only softmax"):
        moe.FusedMoE(8, 2, 256, 128, scoring_func="sigmoid")


def test_fused_experts_shape_assertions(moe):
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    w1 = torch.zeros(2, 32, 48, dtype=torch.bfloat16)
    w2 = torch.zeros(2, 64, 16, dtype=torch.bfloat16)
    tw = torch.zeros(4, 2)
    ids = torch.zeros(4, 2, dtype=torch.int32)
    with pytest.raises(AssertionError, match="Hidden size mismatch"):
        moe.fused_experts(x, w1, w2, None, None, tw, ids)
    w1 = torch.zeros(2, 32, 64, dtype=torch.bfloat16)
    with pytest.raises(AssertionError, match="topk shape mismatch"):
        moe.fused_experts(x, w1, w2, None, None, tw[:, :1], ids)
    with pytest.raises(ValueError, match="Unsupported FusedMoe activation"):
        moe.fused_experts(x, w1, w2, None, None, tw, ids, activation="relu")


def test_fused_experts_takes_ragged_sizes_except_with_e4m3(moe):
    """The reference's Triton kernel masks ragged K and N (for_moe/fused_moe.py:191-205,218-223).
    So does this build for 16-bit and fp32 weights (an element-by-element kernel): such calls pass
    every host check and stop at the device check here.  e4m3 rows move in 16-byte chunks only."""
    tw = torch.zeros(4, 2)
    ids = torch.zeros(4, 2, dtype=torch.int32)
    x = torch.zeros(4, 60, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):           # H = 60
        moe.fused_experts(x, torch.zeros(2, 32, 60, dtype=torch.bfloat16), torch.zeros(2, 60, 16, dtype=torch.bfloat16),
                          None, None, tw, ids)
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):           # I = 12
        moe.fused_experts(x, torch.zeros(2, 24, 64, dtype=torch.bfloat16), torch.zeros(2, 64, 12, dtype=torch.bfloat16),
                          None, None, tw, ids)
    w1 = torch.zeros(2, 32, 68, dtype=torch.bfloat16)[:, :, :64]      # row stride 68
    with pytest.raises(RuntimeError, match="no CPU path"):
        moe.fused_experts(x, w1, torch.zeros(2, 64, 16, dtype=torch.bfloat16), None, None, tw, ids)
    with pytest.raises(RuntimeError, match="no CPU path"):           # fp32, H = 62
        moe.fused_experts(torch.zeros(4, 62), torch.zeros(2, 24, 62), torch.zeros(2, 62, 12), None, None, tw, ids)
    # e4m3: multiples of 16 elements
    f8 = torch.float8_e4m3fn
    with pytest.raises(AssertionError, match="multiples of 16"):
        moe.fused_experts(torch.zeros(4, 72, dtype=torch.bfloat16), torch.zeros(2, 32, 72).to(f8), torch.zeros(2, 72, 16).to(f8),
                          None, None, tw, ids, per_channel_quant=True, w1_scale=torch.ones(2, 32), w2_scale=torch.ones(2, 72))
    # the stride of a dimension of size 1 says nothing: one expert cut out of a larger tensor
    one13 = torch.zeros(3, 32, 64, dtype=torch.bfloat16).as_strided((1, 32, 64), (2051, 64, 1))
    one2 = torch.zeros(3, 64, 16, dtype=torch.bfloat16)[:1]
    with pytest.raises(RuntimeError, match="no CPU path"):
        moe.fused_experts(x, one13, one2, None, None, tw, torch.zeros(4, 2, dtype=torch.int32))
    with pytest.raises(AssertionError, match="global_num_experts"):
        moe.fused_experts(x, torch.zeros(2, 32, 64, dtype=torch.bfloat16), torch.zeros(2, 64, 16, dtype=torch.bfloat16),
                          None, None, tw, ids, global_num_experts=4)
    with pytest.raises(RuntimeError, match="no CPU path"):           # and only then the device check
        moe.fused_experts(x, torch.zeros(2, 32, 64, dtype=torch.bfloat16), torch.zeros(2, 64, 16, dtype=torch.bfloat16),
                          None, None, tw, ids)


def test_block_size_rule_follows_the_activation_dtype(moe):
    cfg = moe.fused_moe.try_get_optimal_moe_config
    w1, w2 = (128, 1536, 2048), (128, 2048, 768)
    assert cfg(w1, w2, 8, None, 768, act_dtype=torch.bfloat16)["BLOCK_SIZE_M"] == 256
    assert cfg(w1, w2, 8, None, 768, act_dtype=torch.float16)["BLOCK_SIZE_M"] == 256
    assert cfg(w1, w2, 8, None, 768, act_dtype=torch.float32)["BLOCK_SIZE_M"] == 64    # fp32 has its own rule
    assert cfg(w1, w2, 8, None, 2048, act_dtype=torch.float32)["BLOCK_SIZE_M"] == 128
    assert cfg(w1, w2, 8, "fp8_w8a8", 384)["BLOCK_SIZE_M"] == 32


def test_plan_and_counters_lie_inside_the_workspace_behind_the_data(moe):
    """Every region of a moe_fused_experts workspace is laid out from
    T*K + E*(block-1), never from the length of the caller's sorted_token_ids buffer:
    the per-block counters and the range table sit behind the intermediates."""
    L = moe._lib.lib()
    for T, H, I, E, K, bs, act, wgt in ((8448, 2048, 768, 128, 8, 256, 2, 2), (256, 2048, 768, 128, 8, 256, 2, 2),
                                        (1, 64, 64, 4, 1, 256, 1, 1), (3000, 512, 256, 16, 4, 512, 2, 3),
                                        (777, 128, 96, 8, 2, 256, 2, 3)):
        total = L.moe_fused_experts_workspace_bytes(T, H, I, E, K, bs, act, wgt)
        b, d = ctypes.c_int64(), ctypes.c_int64()
        n, cap = ctypes.c_int32(), ctypes.c_int32()
        assert L.moe_fused_experts_plan_layout(T, H, I, E, K, bs, act, wgt, ctypes.byref(b), ctypes.byref(d),
                                               ctypes.byref(n), ctypes.byref(cap)) == 1
        sorted_cap = T * K + E * (bs - 1)
        rows = -(-sorted_cap // bs) * bs
        up = lambda v: -(-v // 256) * 256
        data = up(rows * I * 2) + up(T * K * H * 2)
        if wgt == 3:
            data += up(T * H) + up(T * 4) + up(rows * I) + up(rows * 4)
        assert n.value == -(-sorted_cap // 256) and 1 <= cap.value <= n.value
        assert d.value >= data and d.value + 4 * n.value <= b.value and b.value + 256 == total
    # blocks that are not multiples of 256, or fp32, have no plan
    assert L.moe_fused_experts_plan_layout(256, 2048, 768, 128, 8, 32, 2, 2, ctypes.byref(b), ctypes.byref(d),
                                           ctypes.byref(n), ctypes.byref(cap)) == 0
    assert L.moe_fused_experts_plan_layout(256, 2048, 768, 128, 8, 256, 0, 0, ctypes.byref(b), ctypes.byref(d),
                                           ctypes.byref(n), ctypes.byref(cap)) == 0


def test_workloads_are_reproducible_and_skewed(moe):
    wl = moe.workloads
    a = wl.make_inputs(wl.QWEN3_30B_A3B, 256, 1, torch.bfloat16)
    b = wl.make_inputs(wl.QWEN3_30B_A3B, 256, 1, torch.bfloat16)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    assert a[0].shape == (256, 2048) and a[1].shape == (256, 128) and a[1].dtype == torch.float32
    bias = wl.zipf_bias(128, torch.Generator().manual_seed(3))
    assert abs(bias.mean().item()) < 1e-5 and bias.max() - bias.min() > 4.0
    assert wl.layer_flops(8448, wl.QWEN3_30B_A3B) == 637802643456
    assert wl.layer_flops(256, wl.QWEN3_30B_A3B) == 19327352832
    assert wl.layer_bytes(256, wl.QWEN3_30B_A3B, 128) == 1207959552 + 2 * 1048576 + 131072
    shape, x, logits, w13, w2 = wl.make_config("tiny_fp32")
    assert w13.shape == (8, 256, 256) and w2.shape == (8, 256, 128) and x.dtype == torch.float32


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "layered-prefill_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower() or f == "__init__.py" and False, f


@pytest.mark.parametrize("I,E,K,act,wgt,line", [(768, 128, 8, 2, 2, 16), (768, 64, 8, 2, 2, 32), (1024, 32, 4, 1, 1, 48),
                                                (768, 16, 2, 2, 2, 96), (4096, 64, 2, 2, 2, 16), (768, 128, 8, 2, 3, 32),
                                                (1024, 32, 4, 2, 3, 88), (512, 16, 4, 2, 3, 96),
                                                (0, 128, 8, 2, 2, 16), (256, 128, 8, 2, 2, 16), (0, 16, 2, 2, 2, 96)])
def test_layer_block_size_changes_once_at_its_line(moe, I, E, K, act, wgt, line):
    """Blocks of 32 below the line (in routed rows per expert), of 256 from it on."""
    L = moe._lib.lib()
    sizes = [L.moe_layer_block_size(rows * E // K, I, E, K, act, wgt) for rows in range(0, 300)]
    assert sizes == [32] * line + [256] * (300 - line)


@pytest.mark.parametrize("E,H,I,K,weights,layout,last", [
    (128, 2048, 768, 8, 2, 0, 263), (128, 2048, 768, 8, 1, 0, 263), (128, 2048, 768, 8, 2, 1, 255), (32, 2048, 1024, 4, 2, 0, 397),
    (128, 2880, 1440, 4, 2, 0, 597), (32, 2048, 1024, 4, 3, 0, 701), (128, 2880, 1440, 4, 3, 0, 1194), (128, 2048, 768, 8, 3, 0, 511),
    (128, 512, 128, 2, 2, 0, 16108), (6, 24, 40, 2, 2, 0, 287)])
def test_layer_call_changes_its_block_once_at_its_line(moe, E, H, I, K, weights, layout, last):
    """The last batch that streams, by the call's matrix work (and at least 16, e4m3 32, rows per expert; sizes that only
    the register-staged kernels take keep the rule by rows): the workspace a call asks for is that of the block it will use."""
    L, A = moe._lib.lib(), moe._lib.MoeLayerArgs
    act = weights if weights != 3 else 2
    need = lambda T, block: L.moe_layer_workspace_bytes(A(T=T, H=H, I=I, E=E, K=K, act_dtype=act, weight_dtype=weights,
                                                         weight_layout=layout, block_size=block, router_logits=1))
    for T in (1, last // 2, last, last + 1, 2 * last, 16896):
        assert need(T, 32) != need(T, 256)
        assert need(T, 0) == need(T, 32 if T <= last else 256), T


@pytest.mark.parametrize("E,H,I,K,weights,tokens", [
    (128, 2048, 768, 8, 2, (64, 255, 256, 260, 263, 264, 8448)), (16, 4096, 1024, 2, 1, (401, 402, 600, 767, 768)),
    (128, 256, 128, 2, 2, (2048,)), (128, 2880, 1440, 4, 2, (500, 597, 598)), (32, 2048, 1024, 4, 3, (300, 701, 702)),
    (6, 24, 40, 2, 2, (287, 288)), (8, 256, 128, 2, 0, (5, 100, 500))])
def test_a_call_has_the_same_block_size_whichever_way_it_is_entered(moe, E, H, I, K, weights, tokens):
    """The steps enqueued from Python take their block size from ``try_get_optimal_moe_config``, the native call from its
    own arguments: a call of more tokens than the native one takes, or one whose hand-off is checked, must run on the
    kernels of the others.  (The native block shows in the workspace that the call asks for.)"""
    L, A = moe._lib.lib(), moe._lib.MoeLayerArgs
    act = weights if weights != 3 else 2
    dtype = {0: torch.float32, 1: torch.float16, 2: torch.bfloat16}[act]
    for T in tokens:
        for layout, code in moe._lib.WEIGHT_LAYOUT_CODE.items():
            need = lambda block: L.moe_layer_workspace_bytes(A(T=T, H=H, I=I, E=E, K=K, act_dtype=act, weight_dtype=weights,
                                                               weight_layout=code, block_size=block, router_logits=1))
            block = moe.fused_moe.try_get_optimal_moe_config((E, 2 * I, H), (E, H, I), K, "fp8_w8a8" if weights == 3 else None,
                                                             T, act_dtype=dtype, weight_layout=layout)["BLOCK_SIZE_M"]
            assert need(block) == need(0), (T, layout, block)


def test_layer_block_size_of_fp32_is_the_old_rule(moe):
    L = moe._lib.lib()
    for m in (1, 256, 768, 2048, 8448):
        assert L.moe_layer_block_size(m, 768, 128, 8, 0, 0) == L.moe_preferred_block_size(m, 128, 8, 0, 0)


def _hold(module, name, how):
    """Re-registers a parameter as what else a module can hold under that name; returns the tensor it now stands for."""
    t = getattr(module, name).detach()
    if how == "parameter":
        return getattr(module, name)
    if how == "parametrised":
        class Twice(torch.nn.Module):
            def forward(self, w):
                return w + w
        torch.nn.utils.parametrize.register_parametrization(module, name, Twice())
        return t + t
    delattr(module, name)
    if how == "buffer":
        module.register_buffer(name, t)
    else:
        setattr(module, name, t)
    return t


@pytest.mark.parametrize("quantization", [None, "fp8_e4m3"])
@pytest.mark.parametrize("how", ["parameter", "buffer", "attribute", "parametrised"])
def test_layer_takes_weights_however_the_module_holds_them(moe, monkeypatch, how, quantization):
    layer = moe.FusedMoE(4, 2, 32, 16, params_dtype=torch.bfloat16, has_bias=quantization is None,
                         quantization=quantization)
    names = {"w13_weight": 2, "w2_weight": 3}
    if quantization:
        names.update(w13_weight_scale="w1_scale", w2_weight_scale="w2_scale")
        for name, shape in (("w13_weight_scale", (4, 32)), ("w2_weight_scale", (4, 32))):
            layer.register_parameter(name, torch.nn.Parameter(torch.rand(shape), requires_grad=False))
    else:
        names.update(w13_bias="w1_bias", w2_bias="w2_bias")
    for name in names:
        getattr(layer, name).data.fill_(0.25)
    want = {name: _hold(layer, name, how) for name in names}
    seen = []
    monkeypatch.setattr(moe.layer, "fused_topk_experts", lambda *a, **k: seen.append((a, k)) or a[0])
    layer(torch.zeros(3, 32, dtype=torch.bfloat16), torch.zeros(3, 4))
    args, kwargs = seen[0]
    for name, where in names.items():
        assert torch.equal(args[where] if isinstance(where, int) else kwargs[where], want[name]), name


@pytest.mark.parametrize("how", ["parameter", "buffer", "attribute", "parametrised"])
def test_norm_takes_its_weight_however_the_module_holds_it(moe, monkeypatch, how):
    norm = moe.RMSNorm(8)
    want = _hold(norm, "weight", how)

    class Host:
        rms_norm = staticmethod(lambda x, residual, weight, eps: weight)

    class OnGpu:
        is_cuda = True

    monkeypatch.setattr(moe.layer._lib, "host", lambda: Host)
    assert torch.equal(norm(OnGpu()), want)


def test_layer_without_weights_says_so(moe):
    layer = moe.FusedMoE(4, 2, 32, 16, params_dtype=torch.bfloat16)
    del layer.w2_weight
    with pytest.raises(AttributeError, match="w2_weight"):
        layer(torch.zeros(3, 32, dtype=torch.bfloat16), torch.zeros(3, 4))
    quantised = moe.FusedMoE(4, 2, 32, 16, params_dtype=torch.bfloat16, quantization="fp8_e4m3")
    with pytest.raises(RuntimeError, match="before process_weights_after_loading"):
        quantised(torch.zeros(3, 32, dtype=torch.bfloat16), torch.zeros(3, 4))


def test_layer_struct_layout_matches_header(moe):
    text = open(os.path.join(ROOT, "include", "moe_gfx950.h")).read()
    body = text[text.index("typedef struct MoeLayerArgs {") + len("typedef struct MoeLayerArgs {"):text.index("} MoeLayerArgs;")]
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    names = [n.split()[-1].lstrip("*") for decl in body.split(";") if decl.strip() for n in decl.split(",")]
    assert names == [f[0] for f in moe._lib.MoeLayerArgs._fields_]


def test_layer_entry_rejects_bad_calls_without_a_gpu(moe):
    """The C entry of the whole layer checks its sizes, pointers and workspace in front of any launch."""
    L, A = moe._lib.lib(), moe._lib.MoeLayerArgs
    sizes = dict(T=64, H=256, I=128, E=16, K=4, act_dtype=2, weight_dtype=2, logits_dtype=2, w13_stride_e=2 * 128 * 256,
                 w13_stride_n=256, w2_stride_e=256 * 128, w2_stride_n=128)
    tensors = {n: 1 << 20 for n in ("x", "out", "w13", "w2", "router_logits")}   # never followed
    assert L.moe_layer(None) == -1 and L.moe_layer_workspace_bytes(None) == 0
    assert L.moe_layer(A(**{**sizes, "T": 0})) == 0 and L.moe_layer_workspace_bytes(A(**{**sizes, "T": 0})) == 0
    for bad in (dict(T=-1), dict(H=0), dict(E=0), dict(K=0), dict(T=1 << 30), dict(block_size=-1)):
        assert L.moe_layer(A(**{**sizes, **tensors, **bad})) == -1
        assert L.moe_layer_workspace_bytes(A(**{**sizes, **tensors, **bad})) == 0
    for name in ("x", "out", "w13", "w2"):
        assert L.moe_layer(A(**{**sizes, **tensors, name: None})) == -1 and b"null" in L.moe_last_error()
    assert L.moe_layer(A(**{**sizes, **tensors, "router_logits": None})) == -1 and b"topk_ids" in L.moe_last_error()
    need = L.moe_layer_workspace_bytes(A(**sizes, **tensors))
    # without logits the routing's weights and ids come from the caller
    assert need - L.moe_layer_workspace_bytes(A(**{**sizes, **tensors, "router_logits": None})) == 2 * 64 * 4 * 4
    # x's place does not matter, the block size does
    assert L.moe_layer_workspace_bytes(A(**{**sizes, **tensors, "x": (1 << 20) + 2})) == need
    assert L.moe_layer_workspace_bytes(A(**sizes, **tensors, block_size=256)) > need
    assert L.moe_layer(A(**sizes, **tensors)) == -3
    assert L.moe_layer(A(**sizes, **tensors, workspace=1 << 20, workspace_bytes=need - 1)) == -3
    assert L.moe_layer(A(**sizes, **tensors, workspace=(1 << 20) + 128, workspace_bytes=need)) == -3
    assert b"256-byte" in L.moe_last_error()
    assert L.moe_topk_softmax_typed(None, 2, None, None, None, 4, 8, 9, 0, None) == -1
    assert L.moe_topk_softmax_typed(1 << 20, 3, 1 << 20, 1 << 20, None, 4, 8, 2, 0, None) == -1
    assert b"dtype code 3" in L.moe_last_error()
