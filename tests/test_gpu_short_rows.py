"""Forwards of 9 to 64 short rows in one launch (csrc/gemm_few.hip, daxq_linear_short_rows): the bits of the quantisers followed by the GEMM."""
import pytest
import torch

from tests.test_gpu_few_rows import EPS, FMT, FORMS, KIND, _stream, _weight

pytestmark = pytest.mark.gpu


def _longest(L, kind, xf, wf, scheme, round_x, m, n):
    """The longest K, a multiple of 128, that the rule takes."""
    ks = [k for k in range(128, 3073, 128) if L.daxq_linear_short_rows_applies(kind, xf, wf, kind, scheme, round_x, m, n, k)]
    assert ks == list(range(128, 128 * len(ks) + 1, 128))  # no gaps
    return ks[-1] if ks else 0


def _case(fmt, dtype, scheme, m, n, k, round_x=1, pad=0, poison=None, bias=True):
    """(outputs of the one launch, of the separate ones, both as integers, the latter as floats)"""
    from dax_amd import _capi

    L = _capi.lib()
    kind, td = KIND[dtype]
    xf, wf, qmax = FMT[fmt]
    g = torch.Generator("cpu").manual_seed(1000 * m + n + k)
    kp = (k + 127) // 128 * 128
    x = torch.randn(m, k + pad, generator=g)
    x[:, ::37] *= 20
    x[m - 1] *= 0.01
    if poison is not None:
        x[m // 2, k // 3] = poison
    x = x.to(td).to("cuda")
    w = _weight(n, kp, k, wf, g)
    sw = (torch.rand(n, generator=g) * 0.01 + 1e-3).to("cuda")
    b = torch.randn(n, generator=g).to(td).to("cuda") if bias else None
    s_in = torch.tensor([0.037], device="cuda") if scheme == 2 else None
    sp, bp = s_in.data_ptr() if s_in is not None else None, b.data_ptr() if b is not None else None
    got = torch.full((m + 1, n + 3), 7.0, dtype=td, device="cuda")
    _capi.check(L.daxq_linear_short_rows(kind, xf, wf, kind, scheme, round_x, x.data_ptr(), k + pad, sp, w.data_ptr(), kp, sw.data_ptr(), bp,
                                         got.data_ptr(), n + 3, m, n, k, _stream()), "short rows")
    q = torch.zeros(m, kp, dtype=torch.uint8, device="cuda")
    sx = torch.zeros(m, device="cuda")
    part = torch.zeros(256, dtype=torch.int32, device="cuda")
    if scheme == 0:
        rc = L.daxq_act_quant_rows_ex(x.data_ptr(), kind, xf, m, k, k + pad, q.data_ptr(), kp, sx.data_ptr(), qmax, EPS, round_x, _stream())
    elif scheme == 1:
        rc = L.daxq_act_quant_tensor(x.data_ptr(), kind, xf, m, k, k + pad, q.data_ptr(), kp, sx.data_ptr(), None, part.data_ptr(), qmax, EPS,
                                     round_x, _stream())
    else:
        rc = L.daxq_quantize_tensor(x.data_ptr(), kind, xf, m, k, k + pad, sp, q.data_ptr(), kp, sx.data_ptr(), _stream())
    _capi.check(rc, "quantiser")
    want = torch.empty(m, n, dtype=td, device="cuda")
    _capi.check(L.daxq_linear_w8a8(xf, wf, kind, q.data_ptr(), kp, sx.data_ptr(), w.data_ptr(), kp, sw.data_ptr(), bp, want.data_ptr(), n, None, n,
                                   m, n, kp, 0, _stream()), "linear")
    torch.cuda.synchronize()
    assert bool((got[m:] == 7.0).all()) and bool((got[:, n:] == 7.0).all())  # nothing beyond the output is written
    it = torch.int32 if dtype == "fp32" else torch.int16
    return got[:m, :n].contiguous().view(it), want.view(it), want


@pytest.mark.parametrize("scheme", [0, 1, 2])
@pytest.mark.parametrize("fmt,dtype", FORMS)
def test_outputs_are_the_bits_of_the_separate_launches(fmt, dtype, scheme):
    """Every number of rows at which the wavefronts' share or the row blocks change; K of one chunk, ragged against 128 and the longest that
    the rule takes; N ragged against the 32 columns of a workgroup, and beyond 8192; rows at a distance; no bias."""
    from dax_amd import _capi

    L = _capi.lib()
    kind, (xf, wf, _) = KIND[dtype][0], FMT[fmt]
    for m in (9, 15, 16, 17, 24, 25, 31, 32, 33, 40, 41, 48, 57, 64):
        for n in (130, 257, 4100, 8193):
            top = _longest(L, kind, xf, wf, scheme, 1, m, n)
            assert (top == 0) == ((m > 32 and (scheme != 1 or n > 8192)) or (m > 16 and scheme != 1 and n > 8192))
            for k in {8, min(top, 200), max(8, top - 56), top} if top else ():
                got, want, _ = _case(fmt, dtype, scheme, m, n, k, pad=8 * (m % 3), bias=m % 4 != 3)
                assert torch.equal(got, want), (m, n, k)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.0e38])
@pytest.mark.parametrize("scheme", [0, 1, 2])
@pytest.mark.parametrize("fmt,dtype", FORMS)
def test_rows_that_hold_an_infinity_or_a_nan(fmt, dtype, scheme, value):
    """NaN for NaN (its payload is the MFMA's), the other outputs bit for bit."""
    got, want, w = _case(fmt, dtype, scheme, 19, 256, 512, poison=value)
    nan = torch.isnan(w)
    assert torch.equal(got[~nan], want[~nan])
    assert bool(torch.isnan(got.view(w.dtype))[nan].all())


@pytest.mark.parametrize("fmt,dtype,scheme", [("i8", "bf16", 0), ("i8", "fp16", 1), ("i8", "fp32", 0), ("e4m3", "bf16", 1), ("e5m2", "bf16", 1)])
def test_scale_kept_in_fp32(fmt, dtype, scheme):
    for m in (11, 30):
        got, want, _ = _case(fmt, dtype, scheme, m, 300, 488, round_x=0)
        assert torch.equal(got, want)


def test_calls_that_are_not_taken():
    from dax_amd import _capi

    takes = _capi.lib().daxq_linear_short_rows_applies
    for ok in ((0, 0, 0, 0, 0, 1, 9, 1536, 2048), (2, 0, 0, 2, 0, 1, 16, 1, 1536), (0, 1, 1, 0, 2, 1, 32, 8192, 768), (0, 0, 0, 0, 1, 1, 64, 4096, 1024),
               (0, 2, 1, 0, 1, 1, 32, 13824, 256)):
        assert takes(*ok) == 1, ok
    for bad in ((0, 0, 0, 0, 0, 1, 8, 1536, 1536), (0, 0, 0, 0, 0, 1, 33, 1536, 128), (0, 0, 0, 0, 1, 1, 65, 1536, 128), (0, 0, 0, 0, 0, 1, 9, 1536, 2056),
                (2, 0, 0, 2, 0, 1, 9, 1536, 1544), (0, 1, 1, 0, 0, 1, 17, 1536, 776), (0, 0, 0, 0, 0, 1, 9, 8193, 264), (0, 0, 0, 0, 0, 1, 17, 8193, 128),
                (0, 0, 0, 0, 0, 1, 9, 1536, 500), (0, 1, 1, 0, 0, 0, 9, 1536, 512), (0, 1, 1, 0, 0, 1, 9, 127, 512), (0, 1, 2, 0, 0, 1, 9, 1536, 512),
                (1, 1, 1, 1, 0, 1, 9, 1536, 512), (0, 0, 0, 1, 0, 1, 9, 1536, 512), (0, 0, 0, 0, 1, 1, 64, 4095, 1024), (0, 0, 0, 0, 3, 1, 9, 1536, 512)):
        assert takes(*bad) == 0, bad


@pytest.mark.parametrize("fmt", ["int8", "e4m3"])
def test_rows_alone_and_together_and_captured(fmt):
    """A module's rows are the same bits alone, in one launch of many and in a replayed graph."""
    from torch import nn

    from dax_amd.quant.quantization import quantize_dynamic
    from dax_amd.quant.quantization.qconfig import (
        get_dynamic_fp8_per_token_act_per_channel_weight_qconfig, get_dynamic_int8_per_token_act_per_channel_weight_qconfig)

    torch.manual_seed(4)
    model = nn.Sequential(nn.Linear(512, 384)).to("cuda", torch.bfloat16)
    q = get_dynamic_int8_per_token_act_per_channel_weight_qconfig if fmt == "int8" else get_dynamic_fp8_per_token_act_per_channel_weight_qconfig
    quantize_dynamic(model, {"": q()})
    with torch.no_grad():
        x = torch.randn(300, 512, device="cuda", dtype=torch.bfloat16)
        many = model(x)
        for m in (9, 16, 30):
            assert torch.equal(model(x[:m]), many[:m])
        static = x[:20].clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(static)
        for i in range(4):
            static.copy_(x[20 * i: 20 * i + 20])
            graph.replay()
            assert torch.equal(out, many[20 * i: 20 * i + 20])
            assert torch.equal(model(static), out)
            torch.cuda.synchronize()
