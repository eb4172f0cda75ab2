"""The row quantiser at the sizes where it can go wrong: every split of a row over wavefronts, whole and partial chunks,
rows that start on odd addresses, the three element types; and the FP8 bytes it takes without dividing."""
import numpy as np
import pytest
import torch

from oracle import daxq_oracle as O
from tests.util import FINITE_BF16, from_bits

pytestmark = pytest.mark.gpu

FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    import dax_amd.ops as ops

    return ops


def _bytes(t):
    return t.cpu().contiguous().view(torch.uint8).numpy()


# one row length on either side of every change of the kernel's split, then lengths that are no multiple of a chunk
LENGTHS = [1, 7, 8, 9, 504, 512, 520, 1023, 1024, 1032, 1536, 1544, 2041, 2048, 2056, 3072, 3080, 4096, 4104, 6143, 6144,
           6152, 8192, 8200, 10240, 10248, 14336, 14344, 18303, 18432, 18440]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k", LENGTHS)
def test_rows_of_any_length(ops, dtype, k):
    g = torch.Generator().manual_seed(k)
    m = 6
    wide = torch.randn(m, k + 3, generator=g) * torch.tensor([1e-4, 1.0, 30.0, 1.0, 0.0, 3.0])[:, None]
    for x in (wide[:, :k].to(dtype).contiguous(), wide.to(dtype)[:, 3:]):   # the second: rows that start anywhere
        xd = torch.empty(m, x.stride(0), dtype=dtype, device="cuda")[:, :k]
        xd.copy_(x)
        for fmt in ("i8", "e4m3"):
            target = torch.int8 if fmt == "i8" else FP8[fmt]
            qo, so = O.dynamic_quantize(x.contiguous(), (1, k), target, ops.QMAX[fmt], ops.EPS_F32, torch.float32)
            q, s = getattr(ops, "act_quant_" + fmt)(xd)
            assert torch.equal(s.cpu(), so.view(-1))
            np.testing.assert_array_equal(_bytes(q[:, :k]), _bytes(qo))
            assert not q[:, k:].any()
            scale = so.view(-1) * 1.37                                      # the leaf quantiser, rows without padding
            ql = getattr(ops, "quantize_rows_" + fmt)(xd, scale.to("cuda"))
            ref = O.quantize_to_int8(x, scale[:, None]) if fmt == "i8" else O.quantize_to_fp8(x, scale[:, None], target)
            np.testing.assert_array_equal(_bytes(ql), _bytes(ref))


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_fp8_bytes_without_a_division(ops, fmt):
    """FP8 under a scale of any 24 significant bits: x * (1 / s) decides the byte unless it lies within a few fp32 steps of a value
    where the byte changes.  Every finite bf16 element (zeros, subnormals and values beyond the clamp among them) under
    arbitrary scales, scales with few significant bits, powers of two, scales with all bits set and scales at and beyond the
    ends of the range in which the product is used; infinities and NaN; then fp32 elements on and next to the values
    where bytes change."""
    g = torch.Generator().manual_seed(5)
    scales = torch.cat([torch.rand(40, generator=g) * 10 ** (torch.rand(40, generator=g) * 12 - 6),
                        torch.tensor([1.0, 0.5, 2.0 ** -23, 2.0 ** -99, 2.0 ** 99, 2.0 ** -120, 2.0 ** 120, 0.75, 1.25, 3.0, 0.0625 * 7,
                                      float(np.float32(2) - np.float32(2) ** -23), float(np.float32(1) - np.float32(2) ** -24), 1e-38])])
    x = torch.cat([from_bits(FINITE_BF16), torch.tensor([float("inf"), -float("inf"), float("nan")], dtype=torch.bfloat16),
                   torch.zeros(5, dtype=torch.bfloat16)])
    for xs in (x[:32768], x[32768:]):
        for lo in range(0, xs.numel(), 8192):
            row = xs[lo:lo + 8192]
            rows = row.expand(scales.numel(), -1).contiguous()
            q = getattr(ops, "quantize_rows_" + fmt)(rows.to("cuda"), scales.to("cuda"))
            ref = O.quantize_to_fp8(rows, scales[:, None], FP8[fmt])
            nan = torch.isnan(rows.float() / scales[:, None])
            got = q.cpu()
            assert torch.equal(got[~nan], ref.view(torch.uint8)[~nan])
            assert bool(torch.isnan(got.view(FP8[fmt]).float()[nan]).all())
    # fp32 elements: values t at and half-way between the format's, times s, and their fp32 neighbours
    t = torch.arange(0, 127 if fmt == "e4m3" else 124, dtype=torch.uint8).view(FP8[fmt]).float()
    t = torch.cat([t, (t[1:] + t[:-1]) / 2]).double()
    for s in (0.1, 0.003, 1.0 / 3.0, 7.7, 1.0):
        c = (t * s).float().view(torch.int32)[:, None] + torch.arange(-4, 5)
        xf = c.clamp_min(0).to(torch.int32).view(torch.float32).reshape(1, -1)
        xf = torch.cat([xf, -xf], 1)
        sc = torch.tensor([s])
        q = getattr(ops, "quantize_rows_" + fmt)(xf.to("cuda"), sc.to("cuda"))
        assert torch.equal(q.cpu(), O.quantize_to_fp8(xf, sc[:, None], FP8[fmt]).view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,k,pitch", [(1, 8, 8), (1, 5, 5), (3, 7, 9), (255, 33, 33), (300, 1000, 1000), (77, 1001, 1003), (70, 5120, 5128), (2500, 1536, 1536),
                                       (260, 18432, 18432), (5000, 520, 520), (257, 4096, 4104)])
def test_one_scale_for_the_tensor(ops, dtype, m, k, pitch):
    """The abs-max of a tensor over the grid (flat, and rows apart from one another), its last element, first element and a
    place in between as the largest; the scale by the rule of the tensor's type, and bytes, scales and padding against the
    oracle's quantiser of the flattened tensor.  A NaN anywhere makes the scale NaN."""
    g = torch.Generator().manual_seed(m + k)
    base = torch.randn(m, pitch, generator=g).to(dtype)
    for at in ((m - 1, k - 1), (0, 0), (m // 2, k // 3)):
        x = base.clone()
        x[at] = -9.5
        xd = x.to("cuda")[:, :k]
        xc = x[:, :k].contiguous()
        for fmt in ("i8", "e5m2"):
            target = torch.int8 if fmt == "i8" else FP8[fmt]
            qo, so = O.dynamic_quantize(xc.view(1, -1), (1, m * k), target, ops.QMAX[fmt], ops.EPS_F32, torch.float32)
            q, s, s1 = ops.act_quant_tensor(xd, fmt, ops.QMAX[fmt], ops.EPS_F32, True, True)
            assert torch.equal(s1.cpu(), so.view(1)) and torch.equal(s.cpu(), so.view(1).expand(m))
            np.testing.assert_array_equal(_bytes(q[:, :k]), _bytes(qo).reshape(m, k))
            assert q.shape[1] == ops.pad_k(k) and not q[:, k:].any()
            scale = so.view(1) * 0.61                                       # the same with a scale from the caller
            q, s = ops.quantize_tensor(xd, scale.to("cuda"), fmt, False)
            ref = O.quantize_to_int8(xc, scale) if fmt == "i8" else O.quantize_to_fp8(xc, scale, target)
            np.testing.assert_array_equal(_bytes(q), _bytes(ref))
            assert torch.equal(s.cpu(), scale.expand(m))
    x[m // 2, k // 2] = float("nan")
    _, s, s1 = ops.act_quant_tensor(x.to("cuda")[:, :k], "i8", 127.0, ops.EPS_F32, True, True)
    assert bool(torch.isnan(s).all()) and bool(torch.isnan(s1).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,k,pitch", [(128, 512, 512), (129, 512, 512), (2, 64, 64), (2, 63, 63), (128, 65, 67), (64, 513, 515), (42, 1535, 1537),
                                       (43, 1536, 1536), (12, 5115, 5121), (13, 5120, 5120), (3, 18432, 18432), (4, 18431, 18433)])
def test_one_scale_for_a_small_tensor(ops, dtype, m, k, pitch):
    """On either side of 128 pieces of 512 columns, up to which every workgroup takes the abs-max of the matrix itself: the largest
    element in the first and last piece of rows, whole chunks and what they leave over; scale, bytes and padding against the
    oracle's quantiser of the flattened tensor, exactly; an infinity or a NaN in the last element."""
    g = torch.Generator().manual_seed(m + k)
    base = torch.randn(m, pitch, generator=g).to(dtype)
    for n, at in enumerate(((0, 0), (0, k - 1), (m // 2, k // 2), (m - 1, k // 8 * 8 - 1), (m - 1, k - 1))):
        x = base.clone()
        x[at] = -9.5
        x[m - 1, k:] = 100.0  # beyond the rows
        fmt = ("i8", "e4m3", "e5m2")[n % 3]
        target = torch.int8 if fmt == "i8" else FP8[fmt]
        qo, so = O.dynamic_quantize(x[:, :k].reshape(1, -1), (1, m * k), target, ops.QMAX[fmt], ops.EPS_F32, torch.float32)
        q, s, s1 = ops.act_quant_tensor(x.to("cuda")[:, :k], fmt, ops.QMAX[fmt], ops.EPS_F32, True, True)
        assert torch.equal(s1.cpu(), so.view(1)) and torch.equal(s.cpu(), so.view(1).expand(m))
        np.testing.assert_array_equal(_bytes(q[:, :k]), _bytes(qo).reshape(m, k))
        assert q.shape[1] == ops.pad_k(k) and not q[:, k:].any()
    for bad in (float("inf"), float("nan")):
        x[m - 1, k - 1] = bad
        for fmt in ("i8", "e4m3"):
            q, s, s1 = ops.act_quant_tensor(x.to("cuda")[:, :k], fmt, ops.QMAX[fmt], ops.EPS_F32, True, True)
            ref = O.quantize_to_int8 if fmt == "i8" else lambda t, sc: O.quantize_to_fp8(t, sc, FP8["e4m3"])
            assert not bool(torch.isfinite(s).any()) and not bool(torch.isfinite(s1).any())
            if bad == float("inf"):
                np.testing.assert_array_equal(_bytes(q[:, :k])[:-1], _bytes(ref(x[:-1, :k].contiguous(), s1.cpu())))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_every_element_under_scales_near_short_significands(ops, dtype, fmt):
    """All 65536 elements of a 16-bit type: under quotients of short numbers and the format's maximum (calibrated scales), scales
    of any bits, and scales around those with a significand of four bits, where the corrected reciprocal gives way to the
    division.  The bytes are those of an IEEE division."""
    g = torch.Generator().manual_seed(3)
    qmax = torch.tensor(ops.QMAX[fmt])
    bits = [torch.randint(0x3b000000, 0x41000000, (60,), generator=g)]                      # any
    bits.append((torch.rand(40, generator=g) * 90 + 0.01).to(dtype).float().div(qmax).view(torch.int32).long())
    short = 0x3c000000 + torch.randint(0, 80, (12,), generator=g) * (1 << 20)
    bits += [(short[:, None] + torch.tensor([-17, -16, -12, -6, -3, -2, -1, 0, 1, 2, 3, 6, 12, 16, 17])).reshape(-1)]
    bits.append(torch.tensor([2.0 ** -130, 2.0 ** -101, 1.1 * 2.0 ** -90, 1.3 * 2.0 ** -80, 1.7 * 2.0 ** -79, 1.9 * 2.0 ** 99,
                              1.1 * 2.0 ** 100]).view(torch.int32).long())
    scales = torch.cat(bits).to(torch.int32).view(torch.float32)
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).reshape(4, 16384)
    xs, sc = x.repeat(len(scales), 1), scales.repeat_interleave(4)
    q = getattr(ops, "quantize_rows_" + fmt)(xs.to("cuda"), sc.to("cuda"))
    ref = O.quantize_to_fp8(xs, sc[:, None], FP8[fmt])
    nan = torch.isnan(xs)
    np.testing.assert_array_equal(_bytes(q)[~nan.numpy()], _bytes(ref)[~nan.numpy()])
    assert bool(torch.isnan(q.cpu().view(FP8[fmt]).float()[nan]).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,pad", [(897, 0), (1024, 8), (1921, 3), (2049, 0), (3072, 0), (3073, 8), (16384, 0)])
@pytest.mark.parametrize("m", [1, 2, 9, 511, 514, 1031])
def test_one_scale_found_by_the_rows_of_the_quantiser(ops, dtype, k, pad, m):
    """Rows of one to four wavefronts, units of one and two rows, row counts around whole groups of units and of eight units,
    with the largest element anywhere: one reading order for both launches changes neither scale nor bytes."""
    g = torch.Generator("cuda").manual_seed(m + k)
    base = torch.randn(m, k + pad, device="cuda", generator=g).to(dtype)
    s0 = torch.zeros(1, device="cuda")
    for at in ((m - 1, k - 1), (0, 0), (m // 2, k // 2), (max(0, m - 2), 511), (m // 3, k - k % 8 - 1)):
        x = base.clone()
        x[at] = -9.5
        q, s, s1 = ops.act_quant_tensor(x[:, :k], "e4m3", 448.0, ops.EPS_F32, True, True)
        s0.copy_((torch.tensor(9.5).to(dtype) / 448.0).to(torch.float32))
        assert torch.equal(s1, s0) and torch.equal(s, s0.expand(m))
        q1, _ = ops.quantize_tensor(x[:, :k], s0, "e4m3", True)
        assert torch.equal(q, q1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,k,pitch", [(1, 1, 1), (5, 7, 9), (3, 8, 8), (4, 2047, 2047), (3, 2048, 2051), (7, 8193, 8193), (2, 20001, 20001)])
def test_row_statistics_and_weights_in_one_pass(ops, dtype, n, k, pitch):
    """Row minima and maxima with 16-byte loads (chunks, leftover elements, rows that start anywhere; all-negative, zero and
    NaN rows), and the one-pass weight quantiser against them: the same scales and bytes as statistics, scale and leaf
    quantiser one after the other."""
    g = torch.Generator().manual_seed(n * k)
    w = torch.randn(n, pitch, generator=g)
    w[0] = -w[0].abs() - 0.01
    w[-1, k - 1] = 7.5
    w = w.to(dtype).to("cuda")[:, :k]
    lo, hi = ops.row_minmax(w)
    assert torch.equal(lo, w.float().amin(1)) and torch.equal(hi, w.float().amax(1))
    for fmt in ("i8", "e4m3"):
        s = ops.scale_from_minmax(lo, hi, ops.QMAX[fmt])
        q = getattr(ops, "quantize_rows_" + fmt)(w, s)
        q1, s1 = ops.weight_quant(w, fmt, ops.QMAX[fmt], ops.EPS_F32)
        assert torch.equal(s1, s) and torch.equal(q1, q)
    for sign in (1.0, -1.0):
        bad = w.clone()
        bad[n // 2, k // 2] = sign * float("nan")
        lo, hi = ops.row_minmax(bad)
        assert torch.equal(torch.isnan(lo), torch.arange(n, device="cuda") == n // 2) and torch.equal(torch.isnan(hi), torch.isnan(lo))


@pytest.mark.parametrize("fmt", ["i8", "e4m3", "e5m2"])
@pytest.mark.parametrize("k", [8, 64, 504, 512, 520, 1024, 1536, 2048, 2056, 3072, 4104, 6144, 8192, 14336, 18424])
@pytest.mark.parametrize("m", [1, 5])
def test_rows_of_whole_chunks_and_rows_with_a_ragged_end_agree(ops, fmt, k, m):
    """The kernel for rows of whole chunks against the one for any row: a zero column more changes neither scale nor bytes."""
    g = torch.Generator().manual_seed(k + m)
    x = (torch.randn(m, k, generator=g) * 3).bfloat16()
    if m > 1:
        x[1] = 0
        x[2, k // 2] = float("inf")
        x[3, k - 1] = float("nan")
    wide = torch.cat([x, torch.zeros(m, 1, dtype=x.dtype)], dim=1)
    quant = getattr(ops, "act_quant_" + fmt)
    q, s = quant(x.cuda())
    qw, sw = quant(wide.cuda())
    assert torch.equal(s.view(torch.int32), sw.view(torch.int32))
    assert torch.equal(q[:, :k].view(torch.uint8), qw[:, :k].view(torch.uint8)) and not q[:, k:].view(torch.uint8).any()


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("scale", [0.1, 1.0 / 3.0, 0.75, 0.5, 2.0 ** 110])  # arbitrary, bf16, a power of two, one that divides
def test_every_bf16_nan_stays_nan_under_a_scale_from_the_caller(ops, fmt, scale):
    """Every NaN pattern of bf16, both signs, as the only special value of its row, among elements whose quotients lie far
    from every value where a byte changes: the NaN element becomes the format's NaN byte, the others their own bytes."""
    bits = np.concatenate([np.arange(0x7f81, 0x8000), np.arange(0xff81, 0x10000)]).astype(np.uint16)
    m, k = bits.size, 520
    x = torch.full((m, k), 1.296875, dtype=torch.bfloat16)
    at = torch.arange(m) * 37 % k
    x.view(torch.int16)[torch.arange(m), at] = torch.from_numpy(bits.view(np.int16))
    sc = torch.tensor([scale])
    row = O.quantize_to_fp8(torch.full((1, k), 1.296875, dtype=torch.bfloat16), sc[:, None], FP8[fmt]).view(torch.uint8)
    for q in (getattr(ops, "quantize_rows_" + fmt)(x.to("cuda"), sc.expand(m).contiguous().to("cuda")),
              ops.quantize_tensor(x.to("cuda"), sc.to("cuda"), fmt, False)[0]):
        got = q.cpu()
        nan = torch.isnan(got.view(FP8[fmt]).float())
        assert torch.equal(nan, torch.arange(k)[None, :] == at[:, None])
        assert torch.equal(got[~nan], row.expand(m, k)[~nan])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fmt", ["i8", "e4m3", "e5m2"])
@pytest.mark.parametrize("k", [8, 520, 1001, 5120])
def test_an_infinity_in_a_tensor_under_one_scale(ops, dtype, fmt, k):
    """The scale of the tensor is infinite: every finite element is x / inf, a zero with x's sign, and the infinity itself is
    inf / inf: the bytes of the leaf quantiser under that scale."""
    x = torch.randn(5, k, generator=torch.Generator().manual_seed(k)).to(dtype)
    for bad in (float("inf"), -float("inf")):
        x[2, k // 3] = bad
        q, s, s1 = ops.act_quant_tensor(x.to("cuda"), fmt, ops.QMAX[fmt], ops.EPS_F32, True, False)
        assert bool(torch.isinf(s1).all()) and torch.equal(s, s1.expand(5))
        assert torch.equal(q, getattr(ops, "quantize_rows_" + fmt)(x.to("cuda"), s))
        finite = torch.isfinite(x)
        if fmt == "i8":
            assert not q.cpu()[finite].any()
        else:
            assert torch.equal(q.cpu()[finite] & 0x7f, torch.zeros_like(q.cpu()[finite]))
            assert bool(torch.isnan(q.cpu().view(FP8[fmt]).float()[~finite]).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fmt", ["i8", "e4m3", "e5m2"])
@pytest.mark.parametrize("k", [8, 77, 1024, 18440])
def test_weights_that_hold_infinities_and_nans(ops, dtype, fmt, k):
    """The one-pass weight quantiser gives such rows the scale and the bytes of statistics, scale and leaf quantiser, too."""
    w = torch.randn(6, k, generator=torch.Generator().manual_seed(k))
    for row, bad in ((1, float("inf")), (2, -float("inf")), (4, float("nan"))):
        w[row, k // 2] = bad
    w = w.to(dtype).to("cuda")
    s = ops.scale_from_minmax(*ops.row_minmax(w), ops.QMAX[fmt])
    q = getattr(ops, "quantize_rows_" + fmt)(w, s)
    q1, s1 = ops.weight_quant(w, fmt, ops.QMAX[fmt], ops.EPS_F32)
    assert torch.equal(torch.isnan(s1), torch.isnan(s)) and torch.equal(torch.nan_to_num(s1, nan=1.0), torch.nan_to_num(s, nan=1.0))
    if fmt == "i8":
        assert torch.equal(q1, q)
    else:  # (a NaN's sign is not compared)
        a, b = q1.view(FP8[fmt]).float(), q.view(FP8[fmt]).float()
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(q1[~torch.isnan(a)], q[~torch.isnan(a)])


def test_more_rows_than_one_launch_holds(ops):
    """2^25 rows of one wavefront each per launch: scales, bytes and the single scale on either side of the cut."""
    cut, k = 1 << 25, 8
    m = cut + 5
    x = torch.ones(m, k, dtype=torch.bfloat16, device="cuda")
    at = torch.tensor([0, 1, cut - 1, cut, cut + 1, m - 1], device="cuda")
    x[at] = (torch.arange(1, 7, device="cuda")[:, None] * torch.arange(1, k + 1, device="cuda")).bfloat16()
    q, s = ops.act_quant_i8(x[:, :k])
    qs, ss = ops.act_quant_i8(x[at])
    assert torch.equal(q[at], qs) and torch.equal(s[at], ss)
    assert bool((s[7:cut - 7] == s[7]).all())
    del q
    scale = torch.full((m,), 0.25, device="cuda")
    scale[at] = torch.arange(1, 7, device="cuda") * 0.125
    q = ops.quantize_rows_e4m3(x, scale)
    assert torch.equal(q[at], ops.quantize_rows_e4m3(x[at], scale[at]))
    q, s = ops.quantize_tensor(x, scale[:1], "i8", False)
    assert torch.equal(q[at], ops.quantize_tensor(x[at], scale[:1], "i8", False)[0]) and bool((s == scale[0]).all())


def test_more_long_rows_than_one_launch_holds(ops):
    """Rows that take a workgroup each, more of them than the work items of one launch: 2^24 rows of more than 3072 columns."""
    m, k = (1 << 24) + 5, 3080
    if torch.cuda.mem_get_info()[0] < m * k * 3 + (8 << 30):
        pytest.skip("needs 163 GB of free device memory")
    x = torch.empty(m, k, dtype=torch.bfloat16, device="cuda").fill_(1.0)
    scale = torch.full((m,), 0.25, device="cuda")
    at = torch.tensor([0, (1 << 23) - 1, 1 << 23, (1 << 24) - 1, 1 << 24, m - 1], device="cuda")
    x[at] = torch.randn(6, k, device="cuda").bfloat16()
    scale[at] = torch.arange(1, 7, device="cuda") * 0.125
    q = ops.quantize_rows_i8(x, scale)
    assert torch.equal(q[at], ops.quantize_rows_i8(x[at], scale[at]))
    assert bool((q[5:9] == 4).all()) and bool((q[(1 << 24) - 9:(1 << 24) - 5] == 4).all())
    del x, q
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype,m,k", [(torch.bfloat16, 9, 1536), (torch.bfloat16, 40, 1001), (torch.float16, 32, 2048), (torch.bfloat16, 128, 512),
                                       (torch.float32, 64, 1024), (torch.float32, 100, 77)])
@pytest.mark.parametrize("fmt", ["i8", "e4m3", "e5m2"])
def test_bytes_over_the_rows_they_are_made_from(ops, dtype, fmt, m, k):
    """A matrix whose every byte row begins where the row itself does (per-tensor scale; sizes that take one launch elsewhere)"""
    from dax_amd import _capi

    L = _capi.lib()
    kind, width = ops.FLOAT_KIND[dtype], torch.finfo(dtype).bits // 8
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m + k)).to(dtype).to("cuda")
    scale, scratch = torch.zeros(2, m, device="cuda"), torch.zeros(256, dtype=torch.int32, device="cuda")
    apart = torch.zeros(m, width * k, dtype=torch.uint8, device="cuda")
    for i, q in enumerate((apart, x.clone().view(torch.uint8))):
        src = x if i == 0 else q
        _capi.check(L.daxq_act_quant_tensor(src.data_ptr(), kind, ops.FMT[fmt], m, k, k, q.data_ptr(), width * k, scale[i].data_ptr(), None,
                                            scratch.data_ptr(), ops.QMAX[fmt], ops.EPS_F32, 1, torch.cuda.current_stream().cuda_stream), "quant")
        # (only the two launches leave the abs-max of the tensor in the scratch)
        assert bool((scratch != 0).any()) == (i == 1)
        if i == 1:
            assert torch.equal(q[:, :k], apart[:, :k]) and torch.equal(scale[0], scale[1])


@pytest.mark.parametrize("k,m", [(1536, 681), (1536, 683), (1537, 5041), (5120, 205), (5120, 1639), (2560, 3277), (5120, 6557), (1536, 21847), (5120, 26215), (5120, 52429)])
@pytest.mark.parametrize("form", ["token", "one_scale", "tensor"])
def test_matrices_whose_bytes_are_stored_through_the_l2(form, k, m):
    """On either side of the lines between the ways of storing the bytes (1, 8, 32, 128 and 256 MB), numbers of rows that leave the XCDs' ranges
    uneven: the bytes and scales of the whole matrix are those of slices of a few rows, at an address that is a multiple of 8 and at one
    that is not, and nothing around them is written."""
    from dax_amd import _capi

    L = _capi.lib()
    st = torch.cuda.current_stream().cuda_stream
    kp = (k + 127) // 128 * 128
    g = torch.Generator("cuda").manual_seed(k + m)
    x = (torch.randn(m, k, generator=g, device="cuda") * torch.rand(m, 1, generator=g, device="cuda")).to(torch.bfloat16)
    part = torch.empty(256, dtype=torch.int32, device="cuda")
    s1 = torch.tensor([0.0123], device="cuda")

    def quantise(xs, q, sx):
        rows = xs.shape[0]
        if form == "token":
            rc = L.daxq_act_quant_rows(xs.data_ptr(), 0, 0, rows, k, k, q, kp, sx.data_ptr(), st)
        elif form == "one_scale":
            rc = L.daxq_quantize_tensor(xs.data_ptr(), 0, 1, rows, k, k, s1.data_ptr(), q, kp, sx.data_ptr(), st)
        else:
            rc = L.daxq_act_quant_tensor(xs.data_ptr(), 0, 2, rows, k, k, q, kp, sx.data_ptr(), None, part.data_ptr(), 57344.0, 2.0 ** -23, 1, st)
        _capi.check(rc, "quantiser")

    want = torch.zeros(m, kp, dtype=torch.uint8, device="cuda")
    want_s = torch.zeros(m, device="cuda")
    if form == "tensor":  # one scale: the leaf quantiser's bytes under it, in slices
        scale = (x.float().abs().max() / 57344.0).to(torch.bfloat16).float().clamp_min(2.0 ** -23)
        want_s.fill_(scale.item())
        for r in range(0, m, 160):
            n = min(160, m - r)
            _capi.check(L.daxq_quantize_rows(x[r:].data_ptr(), 0, 2, n, k, k, want_s[r:].data_ptr(), want[r:].data_ptr(), kp, st), "rows")
    else:
        for r in range(0, m, 160):
            quantise(x[r:r + 160], want[r:].data_ptr(), want_s[r:])
    for shift in (8, 3):
        buf = torch.full((m * kp + 32,), 0x5A, dtype=torch.uint8, device="cuda")
        sx = torch.full((m + 1,), 7.0, device="cuda")
        quantise(x, buf.data_ptr() + shift, sx)
        torch.cuda.synchronize()
        assert torch.equal(buf[shift:shift + m * kp].view(m, kp), want)
        assert torch.equal(sx[:m], want_s) and sx[m].item() == 7.0
        assert bool((buf[:shift] == 0x5A).all()) and bool((buf[shift + m * kp:] == 0x5A).all())
