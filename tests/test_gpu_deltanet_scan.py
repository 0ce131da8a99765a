"""The bf16 chunk scan's two access paths (v and out in whole pieces, or one
element at a time when their alignment asks for it) and its two column widths:
every pair must give the same bits, since each column's arithmetic is the same."""
import sys

import pytest
import torch

from dan_amd.deltanet import _delta_rule, delta_rule

pytestmark = pytest.mark.gpu


def _inputs(gpu, lengths, hk, hv, dv, seed=11):
    g = torch.Generator().manual_seed(seed)
    n, r = sum(lengths), len(lengths)
    q, k = (torch.randn(n, hk, 128, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    v = torch.randn(n, hv, dv, generator=g).to(torch.bfloat16).to(gpu)
    gate, beta = (-torch.rand(n, hv, generator=g) * 0.2).to(gpu), torch.rand(n, hv, generator=g).to(gpu)
    st = (torch.randn(r, hv, 128, dv, generator=g) * 0.1).to(gpu)
    return q, k, v, gate, beta, lengths, st


def _shifted(x, offset, row_pad):
    """x's values in a buffer that begins `offset` elements past an aligned one, rows `row_pad` elements apart."""
    n, h, d = x.shape
    flat = torch.zeros(offset + n * (h * d + row_pad), dtype=x.dtype, device=x.device)
    out = flat[offset:].as_strided((n, h, d), (h * d + row_pad, d, 1))
    return out


@pytest.mark.parametrize("dv", [32, 64, 128, 256])
@pytest.mark.parametrize("lengths", [[1, 0, 63, 64, 65], [200]])
def test_misaligned_v_and_out(gpu, lengths, dv):
    args = _inputs(gpu, lengths, 2, 4, dv)
    o, f = delta_rule(*args, form="chunk")
    r0 = torch.tensor([sum(lengths[:i]) for i in range(len(lengths))], dtype=torch.int32, device=gpu)
    # (v offset, v row pad, out offset, out row pad), elements: v off 16 bytes, off in the row only, out off 8 bytes, ..
    for vo, vp, oo, op in ((1, 0, 0, 0), (0, 4, 0, 0), (8, 8, 2, 0), (0, 0, 0, 2), (3, 5, 1, 7), (0, 8, 4, 4)):
        print(f"[gpu-case] bf16 scan {lengths} dv {dv}: v +{vo} pad {vp}, out +{oo} pad {op}", flush=True)
        sys.stdout.flush()
        v = _shifted(args[2], vo, vp).copy_(args[2])
        out = _shifted(args[2], oo, op)
        _, f2 = _delta_rule(*args[:2], v, *args[3:], form="chunk", out=out, out_start=r0)
        torch.cuda.synchronize()
        assert torch.equal(out, o) and torch.equal(f2, f)


def test_column_widths_agree(gpu):
    """One run alone (few work groups, 16 columns each) and among many (32): the same bits."""
    lengths = [130, 1, 64] * 13  # 39 runs x 4 heads x 8 column blocks of 16: more groups than two per CU hold
    args = _inputs(gpu, lengths, 4, 4, 128)
    o, f = delta_rule(*args, form="chunk")
    for i in (0, 1, 2, 38):
        a, ln = sum(lengths[:i]), lengths[i]
        print(f"[gpu-case] bf16 scan run {i} of {ln} alone", flush=True)
        o1, f1 = delta_rule(*(x[a:a + ln] for x in args[:5]), [ln], args[6][i:i + 1], form="chunk")
        torch.cuda.synchronize()
        assert torch.equal(o1, o[a:a + ln]) and torch.equal(f1[0], f[i])
