"""The fp32 -> fp16 staging of q and k in one pair of launches against the
definition: x = copy * scale, scale the power of 2 that brings the largest
magnitude into (2^14, 2^15] unless it lies in [2^-6, 2^15]; bit-identical to
staging each tensor alone and to torch's conversion of x / scale."""
import math

import pytest
import torch

from dan_amd.attention import _stage_f16, _stage_f16_pair

pytestmark = pytest.mark.gpu


def scale_of(x):
    m = x.abs().max().item()
    return 1.0 if m == 0 or 2.0 ** -6 <= m <= 2.0 ** 15 else 2.0 ** (math.ceil(math.log2(m)) - 15)


@pytest.mark.parametrize("qs,ks", [((8, 1, 64), (2, 1, 64)), ((8, 384, 64), (2, 384, 64)), ((3, 7, 256), (3, 7, 256)),
                                   ((32, 700, 128), (8, 700, 128)), ((2, 5000, 128), (2, 3, 128))])
@pytest.mark.parametrize("big,small", [(1.0, 1.0), (3e7, 2e-5), (0.0, 1.0)])
def test_pair_equals_the_definition(gpu, qs, ks, big, small):
    print(f"[gpu-case] stage pair {qs} {ks} {big} {small}", flush=True)
    g = torch.Generator().manual_seed(sum(qs))
    # q as the transposed view of a fused token-major buffer, k contiguous
    fused = torch.randn(qs[1], qs[0] + 2, qs[2], generator=g) * big
    q, k = fused.to(gpu)[:, :qs[0]].transpose(0, 1), (torch.randn(ks, generator=g) * small).to(gpu)
    pairs = _stage_f16_pair(q, k)
    alone = _stage_f16(q), _stage_f16(k)
    torch.cuda.synchronize()
    for x, (out, scale), (o1, s1) in zip((q, k), pairs, alone):
        want = scale_of(x)
        assert scale.item() == want == s1.item()
        assert torch.equal(out, (x / want).half()) and torch.equal(out, o1)
