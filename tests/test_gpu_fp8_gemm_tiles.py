"""The e4m3 GEMM's tile shapes (dan_amd/csrc/fp8_gemm.hip: the smallest tile
that gives every CU at most one, 256 x 256 past that) at sizes that choose
each of them on 256 CUs, with ragged rows and columns, K tails of 16 and 48
bytes, K shorter than the ring of stages and an odd number of k-steps.

Bars: those of tests/test_gpu_fp8_gemm.py (every output within the float64
product's bound), raw fp32 sums bit-identical to the matrix-core model, and
the same bits for row-major and tiled operands and for a 300-row call's rows
within a larger call's."""
import pytest
import torch

from dan_amd import quant as DQ
from test_gpu_fp8_gemm import operands, raw_sums_match_model, run_case, say

pytestmark = pytest.mark.gpu

# (m, n) whose smallest tile with at most one per CU (256 CUs) is the named one
SIZES = {"32x32": (33, 48), "32x32 full": (512, 512), "64x32": (300, 1040), "64x64": (520, 1040), "64x128": (1000, 1056),
         "128x128": (2000, 1056), "160x128": (2100, 2064), "192x128": (2500, 2064), "256x128": (3100, 2064),
         "256x256": (4300, 2064)}


@pytest.mark.parametrize("tile", list(SIZES))
@pytest.mark.parametrize("k", [16, 336, 688, 1104])
def test_tile_shapes(gpu, tile, k):
    m, n = SIZES[tile]
    say(f"fp8 GEMM tile {tile}: M {m} N {n} K {k}")
    out_dtype = (torch.bfloat16, torch.float16)[k % 32 == 0]
    xq, wq = run_case(gpu, m, n, k, seed=m + n + k, rowwise=k != 688, out_dtype=out_dtype, with_bias=k != 336,
                      oracle_on_gpu=True)
    r, c = slice(m - min(m, 20), m), slice(n - 48, n)
    raw_sums_match_model(gpu, xq, wq, [(slice(0, min(m, 20)), slice(0, 48)), (r, c), (slice(m // 2, m // 2 + 8), c)])
    g = torch.Generator().manual_seed(k)
    xq, sx, wq, sw = (t.to(gpu) for t in operands(m, n, k, g))
    xt, wt = DQ.tile_codes(xq), DQ.tile_codes(wq)
    ref = DQ.fp8_gemm(xq, sx, wq, sw, None, torch.bfloat16)
    for xa, wa in ((xt, wq), (xq, wt), (xt, wt)):
        y = DQ.fp8_gemm(xa, sx, wa, sw, None, torch.bfloat16)
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
    part = DQ.fp8_gemm(xq[:m // 3 + 1], sx[:m // 3 + 1], wq, sw, None, torch.bfloat16)
    torch.cuda.synchronize()
    assert torch.equal(part, ref[:m // 3 + 1])
