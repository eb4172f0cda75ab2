"""The tiles fitted to launches of one round of workgroups (csrc/gemm_tile_fit.hip): every tile by name at the pair counts and edges
where its pipeline takes another path, and the library's own choice on either side of the lines between it and the other kernels."""
import pytest
import torch

from oracle import daxq_oracle as O

pytestmark = pytest.mark.gpu

TILES = [(64, 64, 5), (64, 96, 4), (64, 128, 6), (64, 192, 4), (128, 96, 5), (128, 160, 4), (128, 224, 3), (192, 192, 3), (256, 96, 3),
         (256, 128, 3), (256, 160, 3)]  # rows, columns, pairs of K slices the LDS holds
OUT = {"bf16": (0, torch.bfloat16), "fp16": (1, torch.float16), "fp32": (2, torch.float32)}


def _operands(m, n, k, fp8, dtype, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    if fp8:
        xq = (torch.randn(m, k, generator=g) * 3).to(torch.float8_e4m3fn).view(torch.uint8)
        wq = (torch.randn(n, k, generator=g) * 0.5).to(torch.float8_e4m3fn).view(torch.uint8)
    else:
        xq = torch.randint(-128, 128, (m, k), generator=g, dtype=torch.int32).to(torch.int8)
        wq = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8)
    sx, sw = torch.rand(m, generator=g) * 0.02 + 1e-3, torch.rand(n, generator=g) * 0.002 + 1e-4
    return xq, wq, sx, sw, torch.randn(n, generator=g).to(dtype)


def _launch(xq, wq, sx, sw, b, fp8, out, kernel, distance=None, e5m2=False):
    """rows behind xq / out's own and columns behind them are checked for writes; distance: elements from one row of outputs to the next"""
    from dax_amd import _capi

    kind, dtype = OUT[out]
    m, k = xq.shape
    n = wq.shape[0]
    d = [t.to("cuda") for t in (xq, wq, sx, sw, b)]
    distance = distance or n + 8
    o = torch.full((m + 1, distance), 7.0, dtype=dtype, device="cuda")
    f = 1 if fp8 else 0
    rc = _capi.lib().daxq_linear_w8a8(2 if e5m2 else f, f, kind, d[0].data_ptr(), k, d[2].data_ptr(), d[1].data_ptr(), k, d[3].data_ptr(), d[4].data_ptr(),
                                      o.data_ptr(), distance, None, 0, m, n, k, kernel, torch.cuda.current_stream().cuda_stream)
    _capi.check(rc, "linear")
    torch.cuda.synchronize()
    assert bool((o[m:] == 7.0).all()) and bool((o[:, n:] == 7.0).all())
    return o[:m, :n].cpu()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_every_tile_at_every_path_of_its_pipeline(tile, fp8):
    """One pair to NS + 4 pairs of K slices (the short form up to NS, then the first pair, steady ones in twos, the odd one behind them)
    on a ragged grid: int8 against the integer oracle, FP8 the bits of the 128x128 tiles (tested against float64 sums elsewhere)."""
    bm, bn, ns = TILES[tile]
    for pairs in range(1, ns + 5):
        m, n, k = bm + 1 + pairs, 2 * bn + 8 * pairs, 128 * pairs
        xq, wq, sx, sw, b = _operands(m, n, k, fp8, torch.bfloat16, 100 * tile + pairs)
        got = _launch(xq, wq, sx, sw, b, fp8, "bf16", 32 + tile)
        if fp8:
            want = _launch(xq, wq, sx, sw, b, True, "bf16", 11 if m >= 128 else 17)
        else:
            want = O.epilogue_int8(O.int_mm(xq, wq), sx.view(-1, 1), sw.view(1, -1), b)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (m, n, k)


@pytest.mark.parametrize("rows", [1, 4, 5, 7, 8, 9, 11, 13, 17, 20, 21])
def test_groups_of_tile_rows(rows):
    """Every tile once, whatever the depth of the tile order's groups: by the launch's tile rows, or named."""
    m, n, k = 64 * rows - (rows > 1), 64 * 7 + 8, 128
    xq, wq, sx, sw, b = _operands(m, n, k, False, torch.bfloat16, rows)
    want = O.epilogue_int8(O.int_mm(xq, wq), sx.view(-1, 1), sw.view(1, -1), b).view(torch.int16)
    for depth in (0, 1, 4, 6, 255):
        assert torch.equal(_launch(xq, wq, sx, sw, b, False, "bf16", 32 | depth << 16).view(torch.int16), want), depth


@pytest.mark.parametrize("out", ["fp16", "fp32"])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tile", [0, 1, 4, 10])  # an even and an odd number of blocks per wavefront in either direction
def test_other_output_types_and_exact_fits(tile, fp8, out):
    """fp16 and fp32 outputs, columns that are no multiple of anything, and a launch of exactly one tile."""
    bm, bn, _ = TILES[tile]
    for m, n in ((bm, bn), (bm + 5, bn + 7)):
        xq, wq, sx, sw, b = _operands(m, n, 1280, fp8, OUT[out][1], m + n)
        other = 5 if not fp8 else 11 if m >= 128 and n >= 128 else 17 if m <= 128 else 32
        got, want = (_launch(xq, wq, sx, sw, b, fp8, out, kernel) for kernel in (32 + tile, other))
        assert torch.equal(got, want)


@pytest.mark.parametrize("out", ["bf16", "fp16"])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_rows_of_outputs_that_start_anywhere(tile, fp8, out):
    """Whole rows of a tile are stored as 16-byte pieces: column counts (and with them row starts, scales and biases) that are a multiple of
    2, 4, 8 or nothing, a tile that is the launch and one that overlaps its neighbours, K in the short and in the pipelined form."""
    bm, bn, ns = TILES[tile]
    other = 5 if not fp8 else 11 if bm >= 128 else 17
    for m, n, pairs in ((bm, bn + 1, 1), (bm + 3, bn + 2, ns + 1), (bm, 2 * bn + 36, ns + 2), (2 * bm - 1, bn, 2)):
        if fp8 and n < 128:
            n += 64
        if fp8 and bm < 128:
            m = min(m, 128)
        xq, wq, sx, sw, b = _operands(m, n, 128 * pairs, fp8, OUT[out][1], m + n + pairs)
        got, want = (_launch(xq, wq, sx, sw, b, fp8, out, kernel) for kernel in (32 + tile, other))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (m, n, pairs)


def test_fp16_sums_of_every_rounded_product():
    """INT8 with fp16 outputs rounds the product to fp16 and adds the bias to that: every fp16 value as the product (an accumulator of
    1, its row's and column's scales), among them subnormal ones and infinity, under biases of all sizes, against torch's two steps."""
    bits = torch.arange(0, 0x7C01, dtype=torch.int32).to(torch.int16).view(torch.float16)
    bits = torch.cat([bits, bits[-1:].repeat(-len(bits) % 64)]).float()
    m = len(bits)
    for bias in (0.0, 1.0, -3.0e-6, 6.0e-8, -0.333, 65504.0, -1234.5):
        n = 64
        xq, wq = torch.zeros(m, 128, dtype=torch.int8), torch.zeros(n, 128, dtype=torch.int8)
        xq[:, 0], wq[:, 0] = 1, 1
        wq[1::2, 0] = -1
        b = torch.full((n,), bias).half()
        got = _launch(xq, wq, bits, torch.ones(n), b, False, "fp16", 32)
        acc = xq.float() @ wq.float().T
        want = ((acc * bits[:, None]).half().float() + b.float()).half()
        same = (got.view(torch.int16) == want.view(torch.int16)) | (got.isnan() & want.isnan())
        assert bool(same.all())


@pytest.mark.parametrize("out", ["bf16", "fp16"])
@pytest.mark.parametrize("fmt", ["int8", "e4m3", "e5m2"])
@pytest.mark.parametrize("k", [384, 640])  # FP8 tiles pipeline from four pairs on
@pytest.mark.parametrize("n", [4088, 4089])
@pytest.mark.parametrize("m", [300, 4300, 5300])  # whole tiles, a last round of quadrants, of halves
def test_ways_of_the_outputs_of_whole_tiles(m, n, k, fmt, out):
    """256x256 tiles store whole rows through the L2 (rows 8256 bytes apart), whole rows (an odd number of elements), or straight from the
    registers (8200 bytes), by the distance of the rows; the same operands all three ways, and in 128x128 tiles."""
    fp8, e5m2 = fmt != "int8", fmt == "e5m2"
    xq, wq, sx, sw, b = _operands(m, n, k, fp8, OUT[out][1], m + n)
    if e5m2:
        xq = xq.view(torch.float8_e4m3fn).float().to(torch.float8_e5m2).view(torch.uint8)
    want = _launch(xq, wq, sx, sw, b, fp8, out, 11 if fp8 else 5, e5m2=e5m2).view(torch.int16)
    for distance in (4100, 4101, 4128):
        assert torch.equal(_launch(xq, wq, sx, sw, b, fp8, out, 8, distance, e5m2).view(torch.int16), want), distance


@pytest.mark.parametrize("k", [128, 256, 384])
@pytest.mark.parametrize("m,n,kernel", [(300, 700, 8), (300, 700, 11), (4300, 4088, 8), (5300, 4088, 8), (4300, 4088, 11)])
def test_short_k_of_fp8_tiles(m, n, kernel, k):
    """Up to three pairs of K slices FP8 tiles of 256x256 (alone, with a last round of quadrants, of halves) and 128x128 do not pipeline,
    and their epilogue's scales go where the last pair's weights were read: every wavefront has to be past them.  Several launches,
    more than a round of workgroups among them, against a fitted tile, whose epilogue keeps its scales in registers."""
    xq, wq, sx, sw, b = _operands(m, n, k, True, torch.bfloat16, m + k)
    want = _launch(xq, wq, sx, sw, b, True, "bf16", 32 + 10)
    for _ in range(4):
        assert torch.equal(_launch(xq, wq, sx, sw, b, True, "bf16", kernel).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("m,n,k", [(64, 16384, 256), (65, 24577, 128), (127, 8200, 1536), (128, 5120, 1024), (129, 4104, 640), (512, 5120, 384),
                                   (2900, 3080, 1024), (4096, 1536, 512), (5000, 64, 512), (5000, 127, 512), (575, 15360, 256), (700, 15360, 256)])
def test_choice_on_either_side_of_the_lines(m, n, k, fp8):
    """The library's own choice: int8 the integer oracle's outputs, FP8 the bits of another kernel of the same sequence of MFMAs."""
    xq, wq, sx, sw, b = _operands(m, n, k, fp8, torch.bfloat16, m + n + k)
    got = _launch(xq, wq, sx, sw, b, fp8, "bf16", 0)
    if fp8:
        want = _launch(xq, wq, sx, sw, b, True, "bf16", 5 if n < 128 else 11 if m >= 128 else 17)
    else:
        want = O.epilogue_int8(O.int_mm(xq, wq), sx.view(-1, 1), sw.view(1, -1), b)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_refused_by_name():
    """A tile larger than the launch, an unknown one, and the accumulator dump are errors of the host, before any launch."""
    from dax_amd import _capi

    L = _capi.lib()
    t = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    p = t.data_ptr()
    st = torch.cuda.current_stream().cuda_stream

    def call(kernel, m, n, acc=None):
        return L.daxq_linear_w8a8(0, 0, 0, p, 128, p, p, 128, p, None, p, n, acc, n, m, n, 128, kernel, st)

    assert call(32, 63, 64) == -1 and call(42, 256, 159) == -1 and call(43, 256, 256) == -1 and call(32, 64, 64, p) == -1
    torch.cuda.synchronize()


def test_rows_and_ranges_of_a_launch():
    """daxq_linear_launch_rows: 64 rows for 33 to 63 of them against many columns, 128 where no fitted tile takes the launch in one round, m
    everywhere else.  daxq_linear_launch_splits: no launch of a forward cuts K."""
    from dax_amd import _capi

    rows, splits = _capi.lib().daxq_linear_launch_rows, _capi.lib().daxq_linear_launch_splits
    for fmt in (0, 1, 2):
        assert [rows(fmt, m, 13824, 5120) for m in (0, 1, 32, 33, 63, 64, 127, 128, 500)] == [0, 1, 32, 64, 64, 64, 127, 128, 500]
        assert [rows(fmt, m, 65536, 1536) for m in (32, 33, 100, 128)] == [32, 128, 128, 128]
        assert [rows(fmt, m, 8192, 1536) for m in (33, 63, 64, 127)] == [33, 63, 64, 127]
    for m, n, k in ((256, 5120, 5120), (128, 5120, 13824), (371, 1536, 13824), (75600, 5120, 5120), (1, 1536, 1536)):
        assert splits(m, n, k) == 1
