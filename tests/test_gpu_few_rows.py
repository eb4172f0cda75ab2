"""The forward of a linear of at most eight rows in one launch (csrc/gemm_few.hip): its outputs are the bits of the quantisers followed by
the GEMM, for every scheme, format and type it takes, and the calls it does not take are refused before any launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

KIND = {"bf16": (0, torch.bfloat16), "fp16": (1, torch.float16), "fp32": (2, torch.float32)}
FMT = {"i8": (0, 0, 127.0), "e4m3": (1, 1, 448.0), "e5m2": (2, 1, 57344.0)}
EPS = 1.1920928955078125e-07
FORMS = [("i8", "bf16"), ("i8", "fp16"), ("i8", "fp32"), ("e4m3", "bf16"), ("e5m2", "bf16")]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _weight(n, kp, k, w_fmt, g):
    if w_fmt == 0:
        w = torch.randint(-127, 128, (n, kp), generator=g, dtype=torch.int32).to(torch.int8).view(torch.uint8)
    else:
        w = (torch.randn(n, kp, generator=g) * 60).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    w[:, k:] = 0
    return w.to("cuda")


def _case(fmt, dtype, scheme, m, n, k, round_x=1, pad=0, poison=None, bias=True, seed=0):
    """(outputs of the one launch, outputs of the separate ones) as integers"""
    from dax_amd import _capi

    L = _capi.lib()
    kind, td = KIND[dtype]
    xf, wf, qmax = FMT[fmt]
    g = torch.Generator("cpu").manual_seed(1000 * m + n + k + seed)
    kp = (k + 127) // 128 * 128
    x = torch.randn(m, k + pad, generator=g)
    x[:, ::37] *= 20
    if poison is not None:
        x[m // 2, k // 3] = poison
    x = x.to(td).to("cuda")
    w = _weight(n, kp, k, wf, g)
    sw = (torch.rand(n, generator=g) * 0.01 + 1e-3).to("cuda")
    b = torch.randn(n, generator=g).to(td).to("cuda") if bias else None
    s_in = torch.tensor([0.037], device="cuda") if scheme == 2 else None
    sp, bp = s_in.data_ptr() if s_in is not None else None, b.data_ptr() if b is not None else None
    got = torch.full((m + 1, n + 3), 7.0, dtype=td, device="cuda")
    assert L.daxq_linear_few_applies(kind, xf, wf, kind, scheme, round_x, m, n, k) == 1
    _capi.check(L.daxq_linear_few(kind, xf, wf, kind, scheme, round_x, x.data_ptr(), k + pad, sp, w.data_ptr(), kp, sw.data_ptr(), bp,
                                  got.data_ptr(), n + 3, m, n, k, _stream()), "few")
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
    """Every number of rows; K of less than a chunk per wavefront, ragged against 128, and up to the limits of the rule; N ragged
    against the 32 columns of a workgroup; rows at a distance; no bias."""
    for m in range(1, 9):
        rows = m if m <= 2 else 4 if m <= 4 else 8
        wide = ((4097, 20488 // rows // 8 * 8), (4100, 40960 // rows - 8), (4100, 40960 // rows), (1000, 24576 // 8)) if m > 2 else ()
        for n, k in ((130, 8), (1000, 520), (257, 1536), (128, 12288 // rows), (4100, min(20480 // rows, 16384)), *wide):
            got, want, _ = _case(fmt, dtype, scheme, m, n, k, pad=8 * (m % 3), bias=m % 4 != 3)
            assert torch.equal(got, want), (m, n, k)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.0e38])
@pytest.mark.parametrize("scheme", [0, 1, 2])
@pytest.mark.parametrize("fmt,dtype", FORMS)
def test_rows_that_hold_an_infinity_or_a_nan(fmt, dtype, scheme, value):
    """The poisoned rows too are those of the separate launches, NaN for NaN (its payload is the MFMA's), the others bit for bit."""
    got, want, w = _case(fmt, dtype, scheme, 5, 256, 1024, poison=value)
    nan = torch.isnan(w)
    assert torch.equal(got[~nan], want[~nan])
    assert bool(torch.isnan(got.view(w.dtype))[nan].all())


@pytest.mark.parametrize("fmt,dtype,scheme", [("i8", "bf16", 0), ("i8", "fp16", 1), ("i8", "fp32", 0), ("e4m3", "bf16", 1), ("e5m2", "bf16", 1)])
def test_scale_kept_in_fp32(fmt, dtype, scheme):
    for m in (1, 6):
        got, want, _ = _case(fmt, dtype, scheme, m, 300, 1480, round_x=0)
        assert torch.equal(got, want)


def test_calls_that_are_not_taken():
    from dax_amd import _capi

    L = _capi.lib()
    takes = L.daxq_linear_few_applies
    assert takes(0, 0, 0, 0, 0, 1, 8, 1, 1536) == 1 and takes(0, 0, 0, 0, 0, 1, 8, 4096, 2560) == 1 and takes(0, 0, 0, 0, 0, 1, 1, 1, 8) == 1
    # int8 beyond 12 KB of rows: of at most 4096 columns against few outputs, at most two rows against many
    assert takes(0, 0, 0, 0, 0, 1, 8, 4095, 3072) == 1 and takes(0, 0, 0, 0, 0, 1, 8, 4095, 3080) == 0 and takes(0, 0, 0, 0, 0, 1, 3, 4095, 4104) == 0
    assert takes(0, 0, 0, 0, 0, 1, 8, 8192, 5120) == 1 and takes(0, 0, 0, 0, 0, 1, 8, 8193, 1544) == 0 and takes(0, 0, 0, 0, 0, 1, 2, 8193, 10240) == 1
    assert takes(0, 1, 1, 0, 0, 1, 3, 4095, 6144) == 1 and takes(0, 1, 1, 0, 0, 1, 8, 8193, 2560) == 1 and takes(0, 1, 1, 0, 0, 1, 2, 4095, 10248) == 0
    for bad in ((0, 0, 0, 0, 0, 1, 9, 1536, 1536), (0, 0, 0, 0, 0, 1, 0, 1536, 1536), (0, 0, 0, 0, 0, 1, 1, 1536, 1540),
                (0, 0, 0, 0, 0, 1, 1, 8192, 16392), (0, 0, 0, 0, 0, 1, 5, 4096, 5128), (0, 0, 0, 1, 0, 1, 1, 1536, 1536),
                (1, 1, 1, 1, 0, 1, 1, 1536, 1536), (0, 1, 2, 0, 0, 1, 1, 1536, 1536), (0, 1, 1, 0, 0, 1, 1, 127, 1536),
                (0, 1, 1, 0, 0, 0, 1, 1536, 1536), (0, 0, 1, 0, 0, 1, 1, 1536, 1536), (0, 0, 0, 0, 3, 1, 1, 1536, 1536)):
        assert takes(*bad) == 0, bad
    t = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    p = t.data_ptr()

    def call(x_off=0, ld_x=128, in_scale=None, scheme=0, w_off=0, ld_w=128, m=1, n=8, k=128):
        return L.daxq_linear_few(0, 0, 0, 0, scheme, 1, p + x_off, ld_x, in_scale, p + w_off, ld_w, p, None, p, n, m, n, k, _stream())

    assert call(ld_x=127) == -1 and call(in_scale=p) == -1 and call(scheme=2) == -1 and call(m=9) == -1 and call(ld_w=1 << 26) == -1
    assert call(x_off=1) == -2 and call(w_off=8) == -2 and call(ld_w=136) == -2
    torch.cuda.synchronize()


@pytest.mark.parametrize("fmt", ["int8", "e4m3"])
def test_forward_captured_and_replayed(fmt):
    """A module's forward of a few rows under capture, replayed on other inputs with eager work in between."""
    from torch import nn

    from dax_amd.quant.quantization import quantize_dynamic
    from dax_amd.quant.quantization.qconfig import (
        get_dynamic_fp8_per_token_act_per_channel_weight_qconfig, get_dynamic_int8_per_token_act_per_channel_weight_qconfig)

    torch.manual_seed(3)
    model = nn.Sequential(nn.Linear(1536, 384)).to("cuda", torch.bfloat16)
    q = get_dynamic_int8_per_token_act_per_channel_weight_qconfig if fmt == "int8" else get_dynamic_fp8_per_token_act_per_channel_weight_qconfig
    quantize_dynamic(model, {"": q()})
    with torch.no_grad():
        xs = [torch.randn(2, 2, 1536, device="cuda", dtype=torch.bfloat16) for _ in range(4)]
        big = model(torch.cat([x.view(-1, 1536) for x in xs]))  # sixteen rows: the separate launches
        static = xs[0].clone()
        model(static)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(static)
        for i, x in enumerate(xs):
            static.copy_(x)
            graph.replay()
            assert torch.equal(out.view(4, 384), big[4 * i: 4 * i + 4])
            assert torch.equal(model(x), out)
            torch.cuda.synchronize()
