"""The conversion of the common case against the general one, which a subclass of the linear takes."""
from functools import partial

import pytest
import torch
from torch import nn

from dax_amd.quant.nn.dynamic import Linear
from dax_amd.quant.quantization import qconfig as Q
from dax_amd.quant.quantization.observer import (DynamicObserverPlaceholder, MinMaxObserver, PerChannelMinMaxObserver,
                                                 plain_settings)

FACTORIES = [getattr(Q, n) for n in dir(Q) if n.startswith("get_") and n != "get_default_dist_profile_qconfig"]


class General(Linear):
    pass


@pytest.mark.parametrize("make", FACTORIES, ids=lambda f: f.__name__)
def test_plain_settings_are_those_of_the_observer(make):
    cfg = make()
    for factory, weight, cls in ((cfg.activation, False, DynamicObserverPlaceholder), (cfg.weight, True, PerChannelMinMaxObserver)):
        got, made = plain_settings(factory, weight), factory()
        assert (got is not None) == (type(made) is cls)
        if got is not None:
            assert (got.dtype, got.qscheme, got.quant_max, got.eps) == (made.dtype, made.qscheme, made.quant_max, float(made.eps))


def test_plain_settings_leave_everything_else_to_the_observer():
    class Own(PerChannelMinMaxObserver):
        pass

    ch = Q.per_channel_symmetric
    for factory in (partial(Own, qscheme=ch), lambda: None, PerChannelMinMaxObserver, partial(PerChannelMinMaxObserver),
                    partial(PerChannelMinMaxObserver, qscheme=ch, ch_axis=1), partial(PerChannelMinMaxObserver, 0, qscheme=ch),
                    partial(PerChannelMinMaxObserver, qscheme=ch, eps=1e-3), partial(PerChannelMinMaxObserver, qscheme=ch, dtype=torch.int32),
                    partial(MinMaxObserver, qscheme=Q.per_tensor_symmetric), partial(DynamicObserverPlaceholder)):
        assert plain_settings(factory, True) is None


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,k,bias,stride", [(1, 1, True, 1), (33, 200, False, 1), (256, 384, True, 1), (64, 128, True, 2)])
@pytest.mark.parametrize("make", [f for f in FACTORIES if "dynamic" in f.__name__ and "channel" in f.__name__], ids=lambda f: f.__name__)
def test_both_conversions_give_one_module(make, n, k, bias, stride, dtype, keep):
    g = torch.Generator("cuda").manual_seed(n + k)
    w = torch.randn(n, k * stride, device="cuda", generator=g).to(dtype)[:, ::stride]
    b = torch.randn(n, device="cuda", generator=g).to(dtype)
    mods = []
    for cls in (Linear, General):
        m = nn.Linear(8, 8, bias=bias)
        m.in_features, m.out_features, m.weight = k, n, nn.Parameter(w)
        if bias:
            m.bias = nn.Parameter(b)
        m.qconfig = make()
        mods.append((m, cls.from_float(m, reserve_float_weight=keep)))
    (f0, q0), (f1, q1) = mods
    assert hasattr(f0, "weight") is hasattr(f1, "weight") is keep
    if q1 is f1:  # not a linear of ours: the float module stays
        assert q0 is f0
        return
    assert type(q0) is Linear and list(q0.state_dict()) == list(q1.state_dict())
    assert q0.__dict__.keys() == q1.__dict__.keys() and q0._fast == q1._fast
    for name in ("in_features", "out_features", "out_dtype", "weight_dtype", "input_dtype", "compute_dtype", "weight_qscheme",
                 "input_qscheme", "training"):
        assert getattr(q0, name) == getattr(q1, name)
    for a, c in zip(q0.state_dict().values(), q1.state_dict().values()):
        assert a.dtype == c.dtype and a.shape == c.shape and a.stride() == c.stride()
        assert torch.equal(a.reshape(-1).view(torch.uint8), c.reshape(-1).view(torch.uint8))
    assert bias == isinstance(q0.bias, nn.Parameter) and (not bias or q0.bias.requires_grad == q1.bias.requires_grad)
    assert (q0._packed is None) == (q1._packed is None) and (q0._sw_vec is None) == (q1._sw_vec is None)
    x = torch.randn(5, k, device="cuda", generator=g).to(dtype)
    assert torch.equal(q0(x), q1(x))
