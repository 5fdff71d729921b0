"""The native host calls (``csrc/host_calls.cpp``) against the Python bodies they stand for: the operators' native CUDA
kernels and the layers' native calls give the same bits, and whatever does not fit them is decided, and refused, by
the general path as before."""

from __future__ import annotations

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _lib():
    from gen_worker_amd import _native

    _native.load()
    assert torch.cuda.is_available()
    yield


def _same(a, b):
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.contiguous().view(torch.uint8),
                                                                      b.contiguous().view(torch.uint8))


def _operands(m, n, k, r, seed=0):
    from gen_worker_amd import synthetic

    layer = synthetic.w4a4_layer(n, k, r, seed_offset=seed)
    x = synthetic.activation(m, k, outlier_frac=0.01, outlier_scale=20.0, seed=seed).to(DEV)
    return x, layer


@pytest.mark.parametrize("m,n,k,r,smooth,bias", [(1, 16, 64, 16, True, True), (77, 272, 448, 32, False, False),
                                                 (300, 384, 640, 64, True, False)])
def test_operator_kernels_equal_the_python_bodies(m, n, k, r, smooth, bias):
    from gen_worker_amd import ops

    x, layer = _operands(m, n, k, r, seed=m)
    sm = layer.smooth.to(DEV) if smooth else None
    one, second = torch.ones((), device=DEV), torch.full((1,), 0.75, device=DEV)
    cg = torch.ops.cozy_gen_worker
    q, s = cg.svdq_quant(x, sm, one, False)
    q0, s0 = ops._svdq_quant_body(x, sm, one, False)
    assert _same(q, q0) and _same(s, s0)
    la = (x @ layer.proj_down.to(DEV)).contiguous()
    args = (q, s, layer.qweight.to(DEV).t().contiguous(), layer.wscales.to(DEV), one, second, la, layer.proj_up.to(DEV),
            layer.bias.to(DEV) if bias else None)
    assert _same(cg.svdq_gemm_w4a4_lora(*args), ops._svdq_gemm_w4a4_lora_body(*args))
    # operands the native kernels leave to the bodies: a bf16 scale, a per-channel second scale in bf16
    q1, s1 = cg.svdq_quant(x, sm, one.to(torch.bfloat16), False)
    assert _same(q1, q0) and _same(s1, s0)
    per = torch.linspace(0.5, 1.5, n, device=DEV).to(torch.bfloat16)
    args = args[:5] + (per,) + args[6:]
    assert _same(cg.svdq_gemm_w4a4_lora(*args), ops._svdq_gemm_w4a4_lora_body(*args))


def test_operator_refusals_are_the_bodies_own():
    from gen_worker_amd import ops

    x, layer = _operands(8, 64, 128, 16)
    one = torch.ones((), device=DEV)
    cg = torch.ops.cozy_gen_worker
    with pytest.raises(ops.SvdqOpError, match="blocked"):
        cg.svdq_quant(x, None, one, True)
    with pytest.raises(ops.SvdqOpError, match="dtype"):
        cg.svdq_quant(x.float(), None, one, False)
    with pytest.raises(ops.SvdqOpError, match="contiguous"):
        cg.svdq_quant(torch.cat([x, x], dim=1)[:, :128], None, one, False)
    with pytest.raises(ops.SvdqOpError, match="one value"):
        cg.svdq_quant(x, None, torch.ones(2, device=DEV), False)
    q, s = cg.svdq_quant(x, None, one, False)
    wq, ws = layer.qweight.to(DEV).t().contiguous(), layer.wscales.to(DEV)
    la, up = torch.zeros(8, 16, device=DEV, dtype=torch.bfloat16), layer.proj_up.to(DEV)
    with pytest.raises(ops.SvdqOpError):
        cg.svdq_gemm_w4a4_lora(q, s, wq, ws, one, torch.ones(1, device=DEV), la[:4], up, None)
    with pytest.raises(ops.SvdqOpError):
        cg.svdq_gemm_w4a4_lora(q, s.float(), wq, ws, one, torch.ones(1, device=DEV), la, up, None)


class _Ops(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


def _awq(n, k, bias=True):
    from gen_worker_amd.awq import AwqPackedLinear

    g = torch.Generator(device=DEV).manual_seed(n + k)
    mod = AwqPackedLinear(k, n, bias=bias, device=DEV)
    with torch.no_grad():
        mod.weight.copy_(torch.randint(0, 256, mod.weight.shape, generator=g, device=DEV, dtype=torch.int32))
        mod.wscales.copy_(torch.rand(mod.wscales.shape, generator=g, device=DEV) * 0.01)
        mod.wzeros.copy_(torch.randn(mod.wzeros.shape, generator=g, device=DEV) * 0.02)
        if bias:
            mod.bias.copy_(torch.randn(n, generator=g, device=DEV))
    return mod


@pytest.mark.parametrize("bias", [True, False])
def test_awq_layer_equals_the_operator(bias):
    from gen_worker_amd import ops

    n, k = 144, 384
    mod = _awq(n, k, bias)
    op = lambda x: torch.ops.cozy_gen_worker.awq_w4a16_mm(  # noqa: E731
        x.reshape(-1, k).contiguous(), mod.weight, mod.wscales, mod.wzeros, mod.bias)
    for m in (0, 1, 5, ops.AWQ_GEMV_MAX_M, ops.AWQ_GEMV_MAX_M + 1):
        x = torch.randn(m, k, device=DEV).to(torch.bfloat16)
        assert _same(mod(x), op(x)), m
    x3 = torch.randn(2, 3, k, device=DEV).to(torch.bfloat16)
    y = mod(x3)
    assert tuple(y.shape) == (2, 3, n) and _same(y.reshape(6, n), op(x3))
    wide = torch.randn(3, 2 * k, device=DEV).to(torch.bfloat16)[:, :k]
    assert _same(mod(wide), op(wide))
    y0 = mod(x3)
    with torch.no_grad():
        mod.weight.data = mod.weight.data.clone() ^ 1   # new storage: read anew by every call
    assert not torch.equal(mod(x3), y0) and _same(mod(x3).reshape(6, n), op(x3))
    mode = _Ops()
    with mode:
        mod(x3)
    assert any("awq_w4a16_mm" in o for o in mode.seen), mode.seen
    with torch.inference_mode():
        assert _same(mod(x3).reshape(6, n), op(x3))
    with pytest.raises(Exception, match="dtype"):
        mod(x3.float())


def _layer(kind, n=272, k=448):
    from gen_worker_amd import synthetic
    from gen_worker_amd.svdq import build_svdq_w4a4_linear
    from gen_worker_amd.w8a8 import build_int8_linear

    if kind == "awq":
        return _awq(n, 384), 384
    if kind == "w8a8":
        w8 = synthetic.w8a8_layer(n, k)
        return build_int8_linear(qweight=w8.qweight, weight_scale=w8.weight_scale, bias=w8.bias, device=DEV), k
    k = 512 if kind == "w4a4_gemv" else k
    _, layer = _operands(4, n, k, 32)
    return build_svdq_w4a4_linear(qweight=layer.qweight, wscales=layer.wscales, smooth=layer.smooth,
                                  proj_down=layer.proj_down, proj_up=layer.proj_up, bias=layer.bias, device=DEV), k


KINDS = ["w4a4", "w4a4_gemv", "w8a8", "awq"]


@pytest.mark.parametrize("kind", ["w4a4", "w8a8"])
def test_layers_native_call_follows_the_module(kind):
    """After the first forward the native call runs; autograd, a mode, another activation, an in-place weight update, a
    LoRA addend and another object or storage under an operand's attribute all leave it for the general path, also one
    of another shape or device, which that path refuses."""
    from gen_worker_amd import synthetic
    from gen_worker_amd.svdq import build_svdq_w4a4_linear
    from gen_worker_amd.w8a8 import build_int8_linear

    n, k = 272, 448
    x, layer = _operands(40, n, k, 32)
    if kind == "w4a4":
        mod = build_svdq_w4a4_linear(qweight=layer.qweight, wscales=layer.wscales, smooth=layer.smooth,
                                     proj_down=layer.proj_down, proj_up=layer.proj_up, bias=layer.bias, device=DEV)
        name = "svdq_forward_fp6"
    else:
        w8 = synthetic.w8a8_layer(n, k)
        mod = build_int8_linear(qweight=w8.qweight, weight_scale=w8.weight_scale, bias=w8.bias, device=DEV)
        name = "w8a8_scaled_mm"
    ref = mod(x)
    native = mod._bound.native
    got = native.run(x, mod.__dict__)
    assert got is not None and _same(got, ref)
    got = native.run(x.reshape(2, 20, k), mod.__dict__)
    assert _same(got, ref.reshape(2, 20, n))
    xr = x.clone().requires_grad_()
    with torch.enable_grad():
        assert native.run(xr, mod.__dict__) is None
    assert native.run(x.float(), mod.__dict__) is None and native.run(x[:, :64], mod.__dict__) is None
    assert native.run(x.cpu(), mod.__dict__) is None and native.run(x[:0], mod.__dict__) is None
    mode = _Ops()
    with mode:
        assert native.run(x, mod.__dict__) is None
        assert _same(mod(x), ref)
    assert any(name in o for o in mode.seen), mode.seen
    if kind == "w4a4":
        with torch.no_grad():
            mod.weight.copy_(mod.weight.flip(0).clone())
        assert native.run(x, mod.__dict__) is None   # the fp6 records are another weight's now
        assert not torch.equal(mod(x), ref)
    else:
        mod.lora_a = torch.randn(8, k, device=DEV).to(torch.bfloat16)
        mod.lora_b = torch.randn(n, 8, device=DEV).to(torch.bfloat16)
        assert native.run(x, mod.__dict__) is None
        assert _same(mod(x), ref + mod._lora_addend(x))
        mod.lora_a = mod.lora_b = None
        assert _same(mod(x), ref)
    bias, data = mod.bias, mod.bias.data
    mod.bias = None
    assert native.run(x, mod.__dict__) is None
    mod.bias = bias
    mod(x)
    native = mod._bound.native
    assert native.run(x, mod.__dict__) is not None
    for other in (torch.cat([data, data]), data.cpu()):
        bias.data = other   # the same Parameter
        assert native.run(x, mod.__dict__) is None
        with pytest.raises(Exception, match="bias|device|cpu"):
            mod(x)
    bias.data = data
    assert native.run(x, mod.__dict__) is not None


@pytest.mark.parametrize("kind", KINDS)
def test_native_calls_run_on_the_current_stream(kind):
    """Queued behind what the caller's stream still has to write, not on the default stream."""
    mod, k = _layer(kind)
    g = torch.Generator(device=DEV).manual_seed(13)
    a, b = (torch.randn(4, k, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    mod(a)
    want = mod(b)
    big = torch.randn(4096, 4096, generator=g, device=DEV)
    x = a.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(4):
            big = torch.sin(big @ big)   # some milliseconds before x is written
        x.copy_(b)
        got = mod(x)
        got2 = got.clone()
    side.synchronize()
    assert _same(got, want) and _same(got2, want)


@pytest.mark.parametrize("m,k", [(1, 64), (3, 448), (4, 512), (5, 576), (130, 1600)])
@pytest.mark.parametrize("smooth", [None, "normal", "subnormal"])
def test_quantizer_without_a_low_rank_product_equals_the_oracle(m, k, smooth):
    """Ends of a wave's four rows and 512 columns; a factor whose reciprocal is not normal takes the division."""
    import numpy as np

    from gen_worker_amd import synthetic
    from oracle import svdq_oracle as O

    bits = lambda t: t.contiguous().view(torch.int16).numpy().view(np.uint16)  # noqa: E731
    x = synthetic.activation(m, k, outlier_frac=0.01, outlier_scale=20.0, seed=m + k)
    sm = None if smooth is None else synthetic.smooth_factor(k, seed=k)
    if smooth == "subnormal":
        sm[k // 2] = 2.0 ** 127
    wide = torch.cat([x, x[:, :8]], dim=1).to(DEV)[:, :k]
    one = torch.ones((), device=DEV)
    want_q, want_s = O.quantize_act_int4(bits(x), None if sm is None else bits(sm))
    from gen_worker_amd import _native as nat

    for a in (x.to(DEV), wide):
        q = torch.empty(m, k // 2, dtype=torch.uint8, device=DEV)
        s = torch.empty(m, k // 64, dtype=torch.float16, device=DEV)
        smd = None if sm is None else sm.to(DEV)
        nat.call("gwa_svdq_quant_int4", a.data_ptr(), a.stride(0), nat.ptr(smd), one.data_ptr(), None, 0, nat.QFMT_INT4,
                 q.data_ptr(), s.data_ptr(), None, m, k, nat.stream_of(a))
        assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(bits(s.cpu()), want_s.view(np.uint16))


@pytest.mark.parametrize("kind", KINDS)
def test_a_trace_records_the_operators(kind):
    """A traced layer computes its output from its input: the native call, which a trace cannot see, leaves the traced
    call to the operators."""
    mod, k = _layer(kind)
    g = torch.Generator(device=DEV).manual_seed(3)
    a, b = (torch.randn(4, k, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    with torch.no_grad():
        mod(a)   # the native call is bound
        traced = torch.jit.trace(mod, (a,))
        assert "cozy_gen_worker" in str(traced.inlined_graph)
        assert _same(traced(a), mod(a)) and _same(traced(b), mod(b))


@pytest.mark.parametrize("kind", KINDS)
def test_a_lazily_negated_activation_is_negated(kind):
    mod, k = _layer(kind)
    x = torch.randn(4, k, generator=torch.Generator(device=DEV).manual_seed(5), device=DEV).to(torch.bfloat16)
    want = mod((-x).contiguous())
    lazy = torch._neg_view(x)
    assert lazy.is_neg() and _same(mod(lazy), want)


@pytest.mark.parametrize("how", ["parameter", "attribute", "parametrized"])
def test_awq_layer_serves_operands_that_are_not_buffers(how):
    import torch.nn.utils.parametrize as P

    mod = _awq(144, 384)
    x = torch.randn(3, 384, generator=torch.Generator(device=DEV).manual_seed(7), device=DEV).to(torch.bfloat16)
    want = mod(x)
    w = mod.weight
    if how == "parameter":
        del mod.weight
        mod.weight = torch.nn.Parameter(w, requires_grad=False)
    elif how == "attribute":
        del mod.weight
        mod.weight = w
    else:
        class Flip(torch.nn.Module):
            def forward(self, t):
                return t ^ 0xFF

        with torch.no_grad():
            mod.weight.copy_(w ^ 0xFF)
            P.register_parametrization(mod, "weight", Flip())
    assert "weight" not in mod._buffers and _same(mod(x), want)


class _Seen(torch.Tensor):
    calls: list = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.calls.append(str(func))
        return super().__torch_function__(func, types, args, kwargs or {})


def test_awq_layer_leaves_operands_the_operator_has_to_see():
    """A weight that vmap batches, a scale that autograd follows, and an operand of a tensor subclass go through the
    operator as before."""
    mod = _awq(144, 384)
    x = torch.randn(3, 384, generator=torch.Generator(device=DEV).manual_seed(7), device=DEV).to(torch.bfloat16)
    want = mod(x)
    both = torch.stack([mod.weight, mod.weight ^ 0x55])
    got = torch.vmap(lambda w: torch.func.functional_call(mod, {"weight": w}, (x,)))(both)
    assert _same(got[0], want)
    assert _same(got[1], torch.func.functional_call(mod, {"weight": both[1].clone()}, (x,)))
    mod.wscales.requires_grad_()
    assert mod(x).requires_grad and _same(mod(x).detach(), want)
    with torch.no_grad():
        assert not mod(x).requires_grad
    mod.wscales.requires_grad_(False)
    mod.wzeros = mod.wzeros.as_subclass(_Seen)
    _Seen.calls.clear()
    assert _same(mod(x).as_subclass(torch.Tensor), want)
    assert any("awq_w4a16_mm" in c for c in _Seen.calls), _Seen.calls


def test_layers_without_the_native_host_calls(monkeypatch):
    """What ``_native.load`` leaves where the extension does not import: the same bits from the Python paths."""
    from gen_worker_amd import ops

    for kind in KINDS:
        mod, k = _layer(kind)
        x = torch.randn(4, k, generator=torch.Generator(device=DEV).manual_seed(11), device=DEV).to(torch.bfloat16)
        mod(x)
        want = mod(x)
        with monkeypatch.context() as mp:
            mp.setattr(ops, "_host", None)
            mp.setattr(ops, "_awq_native", None)
            mod._bound = None
            assert _same(mod(x), want) and _same(mod(x), want), kind
            assert mod._bound is None or mod._bound.native is None


@pytest.mark.parametrize("kind", KINDS)
def test_layers_under_vmap(kind):
    """A batched activation has no storage to hand to the library: the operator's own batching runs."""
    mod, k = _layer(kind)
    x = torch.randn(3, 4, k, generator=torch.Generator(device=DEV).manual_seed(17), device=DEV).to(torch.bfloat16)
    mod(x[0])
    want = torch.stack([mod(t) for t in x])
    assert _same(torch.vmap(mod)(x), want)
