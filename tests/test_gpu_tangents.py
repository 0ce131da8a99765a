"""Forward-mode tangents pass where a launch takes the place of torch's own
operators: attend's prefix saves (clones), the DeltaNet layer's gated norm and
its two narrow projections. Expected: the same operators on the CPU, in fp32
(two bf16 spacings: values and tangents are rounded at each operator)."""
import pytest
import torch
from torch import nn
from torch.autograd import forward_ad

from dan_amd.attention import Batch, attend, segment
from dan_amd.deltanet import _gated_norm, _narrow_pair, gated_rms_norm

pytestmark = pytest.mark.gpu


def dual(t, seed):
    g = torch.Generator().manual_seed(seed)
    return forward_ad.make_dual(t, torch.randn(t.shape, generator=g).to(t))


def close(got, want):
    return ((got.float().cpu() - want.float()).abs() <= 2.0 ** -6 * want.float().abs() + 2.0 ** -6 * want.float().abs().max()).all()


@pytest.mark.parametrize("which", ["k", "v"])
def test_saved_rows_keep_their_tangents(gpu, which):
    print(f"[gpu-case] saves of a dual {which}", flush=True)
    x = torch.randn(90, 12, 64, generator=torch.Generator().manual_seed(1)).bfloat16().to(gpu)
    q, k, v = (t.transpose(0, 1) for t in x.split((8, 2, 2), dim=1))
    segs = Batch([segment(0, [0] * 70 + [1] * 20, None, 33, 0, str(gpu))])
    with torch.no_grad(), forward_ad.dual_level():
        k, v = (dual(t, 2) if name == which else t for name, t in (("k", k), ("v", v)))
        attend(q, k, v, segs, 0)
        for got, t in zip(segs[0].saved[0], (k, v)):
            got, want = forward_ad.unpack_dual(got), forward_ad.unpack_dual(t)
            assert torch.equal(got.primal, want.primal[:, :33])
            assert (got.tangent is None) == (want.tangent is None)
            assert got.tangent is None or torch.equal(got.tangent, want.tangent[:, :33])


@pytest.mark.parametrize("which", ["x", "z", "weight"])
def test_gated_norm_passes_tangents(gpu, which):
    print(f"[gpu-case] gated norm of a dual {which}", flush=True)
    g = torch.Generator().manual_seed(3)
    x, z, weight = (torch.randn(*shape, generator=g).bfloat16() for shape in ((40, 4, 64), (40, 256), (64,)))
    outs = []
    with torch.no_grad(), forward_ad.dual_level():
        for dev, fn in ((gpu, _gated_norm), ("cpu", lambda a, b, w, e: gated_rms_norm(a, b.view(40, 4, 64), w, e).view(40, 256))):
            args = [dual(t.to(dev), 4) if name == which else t.to(dev) for name, t in (("x", x), ("z", z), ("weight", weight))]
            outs.append(forward_ad.unpack_dual(fn(*args, 1e-6)).tangent)
    assert outs[0] is not None and close(outs[0], outs[1])


def test_narrow_projections_pass_tangents(gpu):
    print("[gpu-case] narrow projections of a dual x", flush=True)
    x = torch.randn(40, 256, generator=torch.Generator().manual_seed(5)).bfloat16().to(gpu)
    first, second = (nn.Linear(256, 16, bias=False, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    with torch.no_grad(), forward_ad.dual_level():
        xd = dual(x, 6)
        tangent = forward_ad.unpack_dual(xd).tangent
        for y, m in zip(_narrow_pair(xd, first, second), (first, second)):
            got = forward_ad.unpack_dual(y).tangent
            assert got is not None and close(got, tangent.float().cpu() @ m.weight.float().cpu().T)
