"""Launches of one round of workgroups: 128x128 tiles, 256x128 halves or 256x256 tiles by the number of either and by K.  On either
side of every line the library's own choice gives the bits of the 128x128 tiles (FP8) and of the generic kernel (INT8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (m, n): large tiles / small tiles; 256 CUs
SHAPES = [(260, 8200),    # 66 / 195: small tiles with a CU each
          (516, 6519),    # 78 / 255
          (514, 6600),    # 78 / 260: more than a CU each
          (1100, 3850),   # 80 / 279
          (4096, 2048),   # 128 / 512: two per CU
          (2358, 3239),   # 130 / 494
          (4600, 1800)]   # 144 / 540: a second round of small tiles


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("k", [256, 1920, 2048, 2176])
def test_choice_by_tile_counts(m, n, k):
    import dax_amd.ops as ops
    from dax_amd import _capi

    g = torch.Generator("cuda").manual_seed(m + k)
    sx, sw = torch.rand(m, generator=g, device="cuda") * 0.01, torch.rand(n, generator=g, device="cuda") * 0.01
    bias = torch.randn(n, generator=g, device="cuda")
    for fmt, other, dtype in (("i8", 5, torch.bfloat16), ("i8", 5, torch.float16), ("e4m3", 11, torch.bfloat16)):
        make = lambda rows: (torch.randint(-128, 128, (rows, k), generator=g, dtype=torch.int8, device="cuda") if fmt == "i8" else
                             torch.randn(rows, k, generator=g, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8))
        xq, wq = make(m), make(n)
        got = ops.linear_w8a8(xq, sx, wq, sw, bias.to(dtype), fmt, fmt, dtype)
        try:
            _capi.debug_select_gemm(other)
            ref = ops.linear_w8a8(xq, sx, wq, sw, bias.to(dtype), fmt, fmt, dtype)
        finally:
            _capi.debug_select_gemm(0)
        assert torch.equal(got, ref), (fmt, dtype)
