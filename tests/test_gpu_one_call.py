"""The forward of a quantised linear through the one native call (csrc/torch_linear.cpp): the bits of the general forward
over every scheme, element type and layout it takes, and None wherever the dispatcher would do more than launch kernels."""
import copy
import io
import weakref

import pytest
import torch
from torch import nn

from dax_amd.quant.quantization import convert, prepare, quantize_dynamic
from dax_amd.quant.quantization import qconfig as Q

pytestmark = pytest.mark.gpu

DYNAMIC = {
    "token_i8": Q.get_dynamic_int8_per_token_act_per_channel_weight_qconfig,
    "token_e4m3": lambda: Q.get_dynamic_fp8_per_token_act_per_channel_weight_qconfig(activation_dtype=torch.float8_e4m3fn),
    "token_e5m2": lambda: Q.get_dynamic_fp8_per_token_act_per_channel_weight_qconfig(activation_dtype=torch.float8_e5m2),
    "tensor_i8": Q.get_default_dynamic_int8_qconfig,
    "tensor_e4m3": lambda: Q.get_default_dynamic_fp8_qconfig(activation_dtype=torch.float8_e4m3fn),
    "tensor_e5m2": lambda: Q.get_default_dynamic_fp8_qconfig(activation_dtype=torch.float8_e5m2),
}


def _module(scheme, k, n, dtype, bias, x):
    torch.manual_seed(k + n)
    model = nn.Sequential(nn.Linear(k, n, bias=bias)).to("cuda", dtype)
    if scheme.startswith("static"):
        act = torch.float8_e4m3fn if scheme.endswith("e4m3") else torch.float8_e5m2
        prepare(model, {"": Q.get_fp8_per_channel_weight_qconfig(activation_dtype=act)})
        model(x)
        convert(model)
    else:
        quantize_dynamic(model, {"": DYNAMIC[scheme]()})
    return model[0]


def _general(lin, x):
    """The same forward by way of the custom ops."""
    lin._fast_forward = lambda *a: None
    try:
        return lin(x)
    finally:
        del lin._fast_forward


def _native(lin, x):
    return lin._fast_forward(x, getattr(lin, "act_scale_fp32", False))


@pytest.mark.parametrize("scheme", [*DYNAMIC, "static_e4m3", "static_e5m2"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,k,n,bias", [(1, 128, 16, True), (3, 1000, 40, False), (40, 1024, 264, True), (300, 333, 129, True)])
@torch.no_grad()
def test_bits_of_the_general_forward(scheme, dtype, m, k, n, bias):
    x = torch.randn(m, k, device="cuda").to(dtype)
    lin = _module(scheme, k, n, dtype, bias, x)
    want = _general(lin, x)
    row_wise_16 = dtype != torch.bfloat16 and (scheme.startswith("static") or scheme in ("token_e4m3", "token_e5m2"))
    got = _native(lin, x)
    assert (got is None) == row_wise_16  # a row-wise FP8 module that is not bf16 casts behind the matmul
    assert torch.equal(lin(x), want)
    wide = torch.randn(m, k + 24, device="cuda").to(dtype)
    for y in (x.view(1, m, k), wide[:, 8:8 + k], x.t().contiguous().t(), x[:0]):  # any shape, row stride, strided columns, no rows
        out = lin(y)
        assert out.shape == (*y.shape[:-1], n) and out.dtype == dtype
        assert torch.equal(out, _general(lin, y))


@torch.no_grad()
def test_calls_that_are_not_plain_take_the_op():
    x = torch.randn(24, 256, device="cuda").bfloat16()
    lin = _module("token_i8", 256, 64, torch.bfloat16, True, x)
    want = lin(x)
    assert _native(lin, x) is not None
    assert _native(lin, x.cpu()) is None and _native(lin, x[:, :128]) is None and _native(lin, x.double()) is None
    with pytest.raises(RuntimeError):
        lin(x.cpu())
    with torch.enable_grad():
        assert _native(lin, x.clone().requires_grad_()) is None
    with torch.autograd.forward_ad.dual_level():
        assert _native(lin, torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert _native(lin, x) is None and torch.equal(lin(x), want)
    seen = []

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        assert torch.equal(lin(x), want)
    assert any("daxq.dynamic_linear_i8" in s for s in seen)
    seen.clear()

    class Functions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Functions():
        out = lin(x)
    assert torch.equal(out, want) and any("dynamic_linear_i8" in s for s in seen)
    with torch.inference_mode():
        assert torch.equal(lin(x), want)


@torch.no_grad()
def test_a_lazily_negated_tensor_is_materialised():
    """The bytes of a tensor with the negative bit are those of -x."""
    x = torch.randn(24, 256, device="cuda").bfloat16()
    for scheme in ("token_i8", "tensor_e4m3", "static_e5m2"):
        lin = _module(scheme, 256, 64, torch.bfloat16, True, x)
        neg = torch._neg_view(x)
        assert neg.is_neg() and _native(lin, neg) is None
        assert torch.equal(lin(neg), lin(-x))


@torch.no_grad()
def test_derived_operands_follow_updates_in_place():
    """K = 200: the GEMM reads a zero-padded copy of the weight, which an update of the weight in place makes stale."""
    x = torch.randn(24, 200, device="cuda").bfloat16()
    lin = _module("token_i8", 200, 64, torch.bfloat16, True, x)
    assert _native(lin, x) is not None
    lin.qweight.neg_()
    lin.weight_scale.mul_(2)
    want = _general(lin, x)
    assert torch.equal(_native(lin, x), want)


@torch.no_grad()
def test_capture():
    """On the capture's own stream, which is not the default one."""
    x = torch.randn(24, 256, device="cuda").bfloat16()
    lin = _module("tensor_e4m3", 256, 64, torch.bfloat16, True, x)
    lin(x)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = lin(x)
    for _ in range(3):
        x.mul_(-1)
        want = _general(lin, x)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("k,n", [(0, 8), (16, 0)])
@torch.no_grad()
def test_conversion_of_an_empty_weight(k, n):
    """A weight without elements gives its observer no statistics: the module is built and its scales stay ones."""
    model = nn.Sequential(nn.Linear(k, n, bias=True).to("cuda", torch.bfloat16))
    quantize_dynamic(model, {"": DYNAMIC["token_i8"]()})
    assert model[0].qweight.shape == (n, k) and model[0].weight_scale.shape == (1, n)
    assert bool((model[0].weight_scale == 1).all())


@pytest.mark.parametrize("scheme", [*DYNAMIC, "static_e4m3", "static_e5m2"])
@pytest.mark.parametrize("m", [33, 64, 127])
@torch.no_grad()
def test_buffers_of_more_rows_than_the_call_has(scheme, m):
    """33 to 127 rows against more than 8192 columns run on buffers of 128: the bits of the general forward, for FP8 those of the
    rows in a call of 128; the result has the call's shape and is nobody's view."""
    dtype = torch.float16 if scheme == "token_i8" and m == 64 else torch.bfloat16
    x = torch.randn(128, 520, device="cuda").to(dtype)
    lin = _module(scheme, 520, 8208, dtype, True, x)
    y = _native(lin, x[:m].view(1, m, 520))
    assert y is not None and y.shape == (1, m, 8208) and y.is_contiguous() and not y._is_view()
    assert torch.equal(y[0], _general(lin, x[:m]))
    if not scheme.startswith("tensor"):
        assert torch.equal(y[0], lin(x)[:m])
    with torch.enable_grad():
        y += torch.ones(8208, device="cuda", dtype=dtype, requires_grad=True)
    assert y.requires_grad


@pytest.mark.parametrize("scheme,dtype", [("token_i8", torch.bfloat16), ("token_i8", torch.float16), ("tensor_e4m3", torch.bfloat16),
                                          ("static_e4m3", torch.bfloat16)])
@torch.no_grad()
def test_replaced_state_is_given_back(scheme, dtype):
    """A hook that puts the state elsewhere between forwards (off-loading) gets its device memory back: nothing of the module
    holds the tensors it had."""
    x = torch.randn(32, 1024, device="cuda").to(dtype)
    lin = _module(scheme, 1024, 2048, dtype, True, x)
    want = lin(x)
    assert _native(lin, x) is not None
    kept = {name: t for name, t in (*lin._buffers.items(), *lin._parameters.items()) if t is not None}
    homes = {name: t.detach().cpu() for name, t in kept.items()}
    gone = [weakref.ref(t) for t in kept.values()]
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for name, t in kept.items():
        meta = t.to("meta")
        if name in lin._buffers:
            lin._buffers[name] = meta
        else:
            lin._parameters[name] = nn.Parameter(meta, requires_grad=False)
    del kept, t
    assert all(r() is None for r in gone)
    assert before - torch.cuda.memory_allocated() >= 1024 * 2048
    for name, t in homes.items():
        if name in lin._buffers:
            lin._buffers[name] = t.to("cuda")
        else:
            lin._parameters[name] = nn.Parameter(t.to("cuda"), requires_grad=False)
    assert torch.equal(lin(x), want) and _native(lin, x) is not None


@torch.no_grad()
def test_state_of_another_module_at_the_same_address():
    """K = 200: the zero-padded copy belongs to one tensor, not to the place it lay at; and a copied or unpickled module
    makes its own."""
    x = torch.randn(32, 200, device="cuda").bfloat16()
    lin = _module("tensor_i8", 200, 512, torch.bfloat16, False, x)
    lin(x)
    at = lin.qweight.data_ptr()
    content = -lin.qweight.cpu()
    held = []
    lin._buffers["qweight"] = torch.empty(0, dtype=torch.int8)
    for _ in range(64):  # the allocator hands the freed block out again
        t = torch.empty(content.shape, dtype=torch.int8, device="cuda")
        if t.data_ptr() == at:
            break
        held.append(t)
    t.copy_(content)
    lin._buffers["qweight"] = t
    for module in (lin, copy.deepcopy(lin)):
        want = _general(module, x)
        assert torch.equal(_native(module, x), want)
        assert torch.equal(module._gemm_weight()[:, :200].cpu(), content)
    buf = io.BytesIO()
    torch.save(lin, buf)
    buf.seek(0)
    loaded = torch.load(buf, weights_only=False)
    assert torch.equal(_native(loaded, x), want) and torch.equal(_general(loaded, x), want)


@pytest.mark.parametrize("scheme,dtype", [("token_i8", torch.float16), ("tensor_i8", torch.bfloat16), ("tensor_e5m2", torch.bfloat16),
                                          ("static_e4m3", torch.bfloat16), ("token_i8", torch.bfloat16)])
@torch.no_grad()
def test_settings_changed_after_conversion(scheme, dtype):
    """The module computes with the settings it has when it is called, not with those it was converted with."""
    x = torch.randn(24, 256, device="cuda").to(dtype)
    lin = _module(scheme, 256, 64, dtype, False, x)
    assert lin(x).dtype == dtype
    for other in (torch.float32, torch.float16, dtype):
        lin.out_dtype = other
        assert lin(x).dtype == other and torch.equal(lin(x), _general(lin, x))
    if scheme.startswith("static"):
        lin.input_dtype = torch.float8_e5m2
        assert torch.equal(lin(x), _general(lin, x))
        lin.row_wise_scale = False
        assert torch.equal(lin(x), _general(lin, x))


@torch.no_grad()
def test_a_quantiser_of_the_users_own_is_called():
    """An override of quantize_activation by a subclass, on the module or on the class."""
    from dax_amd.quant.nn.dynamic import Linear

    x = torch.randn(24, 256, device="cuda").half()
    plain = Linear.quantize_activation
    calls = []

    def own(self, input):
        calls.append(input.shape)
        return plain(self, input)

    sub = type("Sub", (Linear,), {"quantize_activation": own})
    lin = _module("token_i8", 256, 64, torch.float16, True, x)
    want = lin(x)
    assert not calls
    lin.__class__ = sub
    assert torch.equal(lin(x), want) and len(calls) == 1
    lin.__class__ = Linear
    lin.quantize_activation = own.__get__(lin)
    assert torch.equal(lin(x), want) and len(calls) == 2
    del lin.quantize_activation
    Linear.quantize_activation = own
    try:
        assert torch.equal(lin(x), want) and len(calls) == 3
    finally:
        Linear.quantize_activation = plain
    assert torch.equal(lin(x), want) and len(calls) == 3


@pytest.mark.parametrize("scheme,k", [("token_i8", 256), ("tensor_i8", 200), ("static_e4m3", 256), ("static_e4m3", 200)])
@torch.no_grad()
def test_state_that_is_no_parameter_or_buffer(scheme, k):
    """A wrapper may keep the state as plain attributes (a sharding framework's flat parameter) or compute it
    (torch.nn.utils.parametrize): the module reads it by name."""
    x = torch.randn(24, k, device="cuda").bfloat16()
    lin = _module(scheme, k, 64, torch.bfloat16, True, x)
    want = lin(x)
    for name in ("qweight", "weight_scale", "bias", "input_scale"):
        if name in lin._parameters or name in lin._buffers:
            t = getattr(lin, name).detach()
            delattr(lin, name)
            setattr(lin, name, t)
    assert "qweight" not in lin._parameters and "qweight" not in lin._buffers
    assert torch.equal(lin(x), want) and torch.equal(_native(lin, x), want)


@torch.no_grad()
def test_a_scale_of_the_other_form():
    """A per-tensor weight scale replaced by one per channel and back: the vector made from the scalar does not stay."""
    x = torch.randn(24, 256, device="cuda").bfloat16()
    lin = _module("tensor_i8", 256, 64, torch.bfloat16, True, x)
    scalar, per_channel = lin.weight_scale, torch.rand(1, 64, device="cuda") + 0.5
    for s in (scalar, per_channel, scalar, scalar * 2, per_channel):
        lin.weight_scale = s
        got = _native(lin, x)
        assert got is not None and torch.equal(got, _general(lin, x))
        vector = lin._weight_scale_vector()
        assert torch.equal(vector, s.reshape(-1).expand(64))


@torch.no_grad()
def test_settings_that_a_subclass_computes():
    """An out_dtype that is a property, and a module saved with a quantiser of the user's own."""
    from dax_amd.quant.nn.dynamic import Linear

    x = torch.randn(24, 256, device="cuda").half()
    lin = _module("token_i8", 256, 64, torch.float16, False, x)
    want = lin(x)
    del lin.out_dtype
    lin.__class__ = type("Sub", (Linear,), {"out_dtype": property(lambda self: torch.float16)})
    assert torch.equal(lin(x), want) and torch.equal(_native(lin, x), want)
    lin.__class__ = type("Own", (Linear,), {"out_dtype": torch.float16, "quantize_activation": lambda self, x: Linear.quantize_activation(self, x)})
    assert torch.equal(lin(x), want) and _native(lin, x) is None
    lin.__class__ = Linear
    lin.out_dtype = torch.float16
    buf = io.BytesIO()
    torch.save(lin, buf)


@pytest.mark.parametrize("scheme", ["token_i8", "tensor_e4m3", "static_e4m3"])
@torch.no_grad()
def test_conversion_prepares_the_first_forward(scheme):
    """What the native call needs besides the state is there before the first forward, and that forward makes nothing anew."""
    x = torch.randn(24, 200, device="cuda").bfloat16()
    lin = _module(scheme, 200, 64, torch.bfloat16, True, x)
    ready = lin._fast, lin._packed, lin._sw_vec
    assert ready[0] is not None and ready[1] is not None
    lin(x)
    assert all(a is b for a, b in zip(ready, (lin._fast, lin._packed, lin._sw_vec)))
