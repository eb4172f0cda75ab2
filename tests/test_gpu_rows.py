"""The GEMM for a handful of rows: every row block count and ring depth, ragged in both dimensions, K from one step to more
steps than the ring holds, every output type and operand format.  INT8 against the integer oracle's epilogue, bit for bit;
FP8 the same bits as the tiled kernel (an output row does not depend on how many rows the launch has)."""
import pytest
import torch

from oracle import daxq_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture()
def select():
    from dax_amd import _capi

    yield _capi.debug_select_gemm
    _capi.debug_select_gemm(0)


# n on either side of the widths at which the form changes (2048, 4096, 8192) and ragged; k / 128 = 1 .. 44 steps
SHAPES = [(5, 128), (16, 256), (17, 384), (130, 640), (264, 1408), (133, 1536), (2048, 1280), (2052, 1152), (4095, 512), (4097, 640),
          (8192, 256), (8200, 384), (520, 5632)]
ROWS = [1, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 100, 127, 128]


@pytest.mark.parametrize("n,k", SHAPES)
def test_rows_int8(select, n, k):
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(n + k)
    xq = torch.randint(-128, 128, (128, k), generator=g, dtype=torch.int8)
    wq = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    sx, sw = torch.rand(128, generator=g) * 0.01, torch.rand(n, generator=g) * 0.01
    acc = O.int_mm(xq, wq)
    select(17)
    xd, wd = xq.to("cuda"), wq.to("cuda")
    for i, m in enumerate(ROWS):
        dtype = (torch.bfloat16, torch.float16, torch.float32)[i % 3]
        bias = torch.randn(n, generator=g).to(dtype) if i % 2 else None
        ref = O.epilogue_int8(acc[:m], sx[:m, None], sw, bias, out_dtype=dtype)
        y = ops.linear_w8a8(xd[:m], sx[:m].to("cuda"), wd, sw.to("cuda"), None if bias is None else bias.to("cuda"), "i8", "i8", dtype)
        assert y.dtype == dtype and torch.equal(y.cpu(), ref), (m, dtype)


@pytest.mark.parametrize("x_fmt,w_fmt", [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")])
@pytest.mark.parametrize("n,k", [s for s in SHAPES if s[0] >= 128])
def test_rows_fp8_bits_of_the_tiled_kernel(select, n, k, x_fmt, w_fmt):
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(n * 3 + k)
    f8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
    xq = torch.randn(128, k, generator=g).to(f8[x_fmt]).view(torch.uint8).to("cuda")
    wq = torch.randn(n, k, generator=g).to(f8[w_fmt]).view(torch.uint8).to("cuda")
    sx, sw = torch.rand(128, generator=g).to("cuda"), torch.rand(n, generator=g).to("cuda")
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        bias = torch.randn(n, generator=g).to(dtype).to("cuda")
        select(11)
        ref = ops.linear_w8a8(xq, sx, wq, sw, bias, x_fmt, w_fmt, dtype)
        select(17)
        for m in ROWS:
            assert torch.equal(ops.linear_w8a8(xq[:m], sx[:m], wq, sw, bias, x_fmt, w_fmt, dtype), ref[:m]), (m, dtype)


def test_rows_outputs_as_a_slice_of_a_wider_buffer():
    """Strided operands and output through the C ABI: nothing outside the M x N outputs is touched."""
    import dax_amd.ops as ops
    from dax_amd import _capi

    g = torch.Generator().manual_seed(3)
    m, n, k = 19, 83, 384
    xq = torch.randint(-128, 128, (m, k + 128), generator=g, dtype=torch.int8).to("cuda")[:, :k]
    wq = torch.randint(-128, 128, (n, k + 256), generator=g, dtype=torch.int8).to("cuda")[:, :k]
    sx, sw = torch.rand(m, generator=g).to("cuda"), torch.rand(n, generator=g).to("cuda")
    out = torch.full((m + 2, n + 10), 7.0, dtype=torch.bfloat16, device="cuda")
    view = out[1:m + 1, 3:n + 3]
    _capi.check(_capi.lib().daxq_linear_w8a8(0, 0, 0, xq.data_ptr(), xq.stride(0), sx.data_ptr(), wq.data_ptr(), wq.stride(0), sw.data_ptr(), None,
                                             view.data_ptr(), out.stride(0), None, 0, m, n, k, 17, torch.cuda.current_stream().cuda_stream), "rows")
    ref = O.epilogue_int8(O.int_mm(xq.cpu(), wq.cpu()), sx.cpu()[:, None], sw.cpu(), None)
    assert torch.equal(view.cpu(), ref)
    view.fill_(7.0)
    assert bool((out == 7.0).all())


# more than 128 rows: outputs of 16 x 16 blocks on either side of every count at which the form or the kernel changes, ragged in
# both dimensions, fewer than 128 columns, K below and above 2048
MANY = [(129, 40, 256), (130, 800, 384), (512, 256, 2176), (513, 260, 256), (640, 250, 640), (641, 256, 2176), (1023, 255, 2048), (1040, 257, 128),
        (200, 1570, 2176), (300, 1715, 256), (257, 1936, 1920), (16, 1, 128), (5000, 17, 256), (2047, 127, 1152), (6001, 100, 384)]


@pytest.mark.parametrize("m,n,k", MANY)
def test_few_outputs_of_many_rows(m, n, k):
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(m + n)
    sx, sw = torch.rand(m, generator=g) * 0.01, torch.rand(n, generator=g) * 0.01
    xq = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int8)
    wq = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    acc = O.int_mm(xq, wq)
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        bias = torch.randn(n, generator=g).to(dtype)
        y = ops.linear_w8a8(xq.to("cuda"), sx.to("cuda"), wq.to("cuda"), sw.to("cuda"), bias.to("cuda"), "i8", "i8", dtype)
        assert torch.equal(y.cpu(), O.epilogue_int8(acc, sx[:, None], sw, bias, out_dtype=dtype)), dtype
    # FP8: an output row's bits do not depend on how many rows the launch has (128 at a time is the same kernel's other form)
    x8 = torch.randn(m, k, generator=g).to(torch.float8_e4m3fn).view(torch.uint8).to("cuda")
    w8 = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn).view(torch.uint8).to("cuda")
    sxd, swd = sx.to("cuda"), sw.to("cuda")
    y = ops.linear_w8a8(x8, sxd, w8, swd, None, "e4m3", "e4m3", torch.bfloat16)
    parts = [ops.linear_w8a8(x8[i:i + 128], sxd[i:i + 128].contiguous(), w8, swd, None, "e4m3", "e4m3", torch.bfloat16) for i in range(0, m, 128)]
    assert torch.equal(y, torch.cat(parts))


@pytest.mark.parametrize("n,k,m", [(64, 5120, 6600), (1, 384, 300), (127, 13824, 700), (40, 256, 50000)])
def test_fp8_rows_of_a_narrow_layer_do_not_depend_on_the_others(n, k, m):
    """Fewer than 128 output channels: the same bits for a row alone, among a few and in a launch of many."""
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(torch.float8_e4m3fn).view(torch.uint8).to("cuda")
    w = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn).view(torch.uint8).to("cuda")
    sx, sw = torch.rand(m, generator=g).to("cuda"), torch.rand(n, generator=g).to("cuda")
    y = ops.linear_w8a8(x, sx, w, sw, None, "e4m3", "e4m3", torch.float32)
    for rows in (1, 16, 17, 128, 129, m // 2):
        assert torch.equal(ops.linear_w8a8(x[:rows], sx[:rows], w, sw, None, "e4m3", "e4m3", torch.float32), y[:rows]), rows


@pytest.mark.parametrize("fmt", ["i8", "e4m3", "e5m2"])
@pytest.mark.parametrize("n,k", [(130, 640), (264, 1408), (2052, 1152)])
def test_accumulators_beside_the_outputs_of_few_rows(n, k, fmt):
    """The form that returns the accumulators as well gives the outputs of the plain form, bit for bit, and the accumulators
    they come from."""
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(n)
    if fmt == "i8":
        x, w = (torch.randint(-128, 128, s, generator=g, dtype=torch.int8).to("cuda") for s in ((300, k), (n, k)))
    else:
        f8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}[fmt]
        x, w = (torch.randn(*s, generator=g).to(f8).view(torch.uint8).to("cuda") for s in ((300, k), (n, k)))
    sx, sw = torch.rand(300, generator=g).to("cuda"), torch.rand(n, generator=g).to("cuda")
    for m in (1, 17, 64, 100, 127, 128, 300):
        if m > 128 and n > 1000:  # (2000 blocks of 16 x 16 and more: the tiled kernels)
            continue
        for dtype in (torch.bfloat16, torch.float16, torch.float32):
            bias = torch.randn(n, generator=g).to(dtype).to("cuda")
            y = ops.linear_w8a8(x[:m], sx[:m], w, sw, bias, fmt, fmt, dtype)
            ya, acc = ops.linear_w8a8_acc(x[:m], sx[:m], w, sw, bias, fmt, fmt, dtype)
            assert torch.equal(y, ya), (m, dtype)
            if dtype == torch.float32:
                assert torch.equal(y, acc.float() * sx[:m, None] * sw + bias), m
            if fmt == "i8":
                assert torch.equal(acc.cpu(), O.int_mm(x[:m].cpu(), w.cpu()))


@pytest.mark.parametrize("x_fmt,w_fmt", [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")])
@pytest.mark.parametrize("n,k", [(5120, 640), (5121, 128), (5128, 512), (6000, 1408)])
def test_fp8_bits_of_the_tiled_kernel_at_65_to_128_rows(select, n, k, x_fmt, w_fmt):
    """Either side of the width from which four row blocks share a wavefront, K from one step to more than its ring holds."""
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(n * 3 + k)
    f8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
    xq = torch.randn(128, k, generator=g).to(f8[x_fmt]).view(torch.uint8).to("cuda")
    wq = torch.randn(n, k, generator=g).to(f8[w_fmt]).view(torch.uint8).to("cuda")
    sx, sw = torch.rand(128, generator=g).to("cuda"), torch.rand(n, generator=g).to("cuda")
    select(11)
    ref = ops.linear_w8a8(xq, sx, wq, sw, None, x_fmt, w_fmt, torch.float32)
    select(0)
    for m in (64, 65, 80, 113, 127, 128):
        assert torch.equal(ops.linear_w8a8(xq[:m], sx[:m], wq, sw, None, x_fmt, w_fmt, torch.float32), ref[:m]), m


@pytest.mark.parametrize("m", [64, 65, 100, 127, 128])
@pytest.mark.parametrize("n,k", [(5120, 8960), (4104, 13704), (8192, 5632)])
def test_int8_rows_against_a_large_weight(m, n, k):
    """K cut into ranges on 128 rows of the op's own buffers: the outputs of the first m, bit for bit."""
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(m, k, generator=g).bfloat16()
    wq = torch.randint(-128, 128, (n, ops.pad_k(k)), generator=g, dtype=torch.int8)
    wq[:, k:] = 0
    sw, bias = torch.rand(n, generator=g) * 0.01, torch.randn(n, generator=g).bfloat16()
    xq, sx = O.dynamic_quantize(x, (1, k), torch.int8, 127.0, ops.EPS_F32, torch.float32)
    ref = O.epilogue_int8(O.int_mm(xq, wq[:, :k].contiguous()), sx.view(-1, 1), sw, bias)
    args = [t.to("cuda") for t in (x, wq, sw, bias)]
    for _ in range(2):  # (the second launch finds the workspace's counters as the first left them)
        y = ops.dynamic_linear_i8(*args)
        assert y.shape == (m, n) and torch.equal(y.cpu(), ref)


@pytest.mark.parametrize("m", [33, 48, 64, 65, 100, 127])
@pytest.mark.parametrize("n,k", [(8200, 1408), (13824, 640)])
def test_33_to_127_rows_against_many_columns(m, n, k):
    """The library's own choice on buffers of just m rows: INT8 against the oracle's epilogue, FP8 the bits of the first m rows
    of a launch of 128, with and without the accumulators."""
    import dax_amd.ops as ops

    g = torch.Generator().manual_seed(m + n)
    sx, sw = torch.rand(128, generator=g) * 0.01, torch.rand(n, generator=g) * 0.01
    xq = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int8)
    wq = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    sxd, swd = sx.to("cuda"), sw.to("cuda")
    y = ops.linear_w8a8(xq.to("cuda"), sxd[:m], wq.to("cuda"), swd, None, "i8", "i8", torch.float16)
    assert torch.equal(y.cpu(), O.epilogue_int8(O.int_mm(xq, wq), sx[:m, None], sw, None, out_dtype=torch.float16))
    for x_fmt, w_fmt in (("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")):
        f8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
        x = torch.randn(128, k, generator=g).to(f8[x_fmt]).view(torch.uint8).to("cuda")
        w = torch.randn(n, k, generator=g).to(f8[w_fmt]).view(torch.uint8).to("cuda")
        for dtype in (torch.bfloat16, torch.float16, torch.float32):
            ref = ops.linear_w8a8(x, sxd, w, swd, None, x_fmt, w_fmt, dtype)
            assert torch.equal(ops.linear_w8a8(x[:m], sxd[:m], w, swd, None, x_fmt, w_fmt, dtype), ref[:m]), (x_fmt, w_fmt, dtype)
            assert torch.equal(ops.linear_w8a8_acc(x[:m], sxd[:m], w, swd, None, x_fmt, w_fmt, dtype)[0], ref[:m])
