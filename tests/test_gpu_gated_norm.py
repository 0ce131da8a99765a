"""The DeltaNet layer's gated RMS norm kernel (dan_gdn_gated_norm) against the
eager ops of dan/fused.py:52-56 (dan_amd.deltanet.gated_rms_norm) on the CPU.

Bars: both round at the same places, so an output can differ only where the
sum's order or the last ulps of rsqrt and silu move a rounding: at least
99.9 % of the values have the same bits, and each is within three spacings of
the type at its magnitude (one rounding of x rsqrt, one of the product with
the weight, one at the store)."""
import sys

import pytest
import torch

from dan_amd.deltanet import _gated_norm, gated_rms_norm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,hv,dv", [(1, 1, 32), (7, 3, 32), (33, 4, 64), (257, 16, 128), (5, 1, 128), (61, 2, 256), (1, 32, 256)])
def test_gated_norm_matches_eager(gpu, dtype, n, hv, dv):
    print(f"[gpu-case] gated norm {dtype} {n} x {hv} x {dv}", flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(n + hv + dv)
    x = (torch.randn(n, hv, dv, generator=g) * torch.logspace(-4, 2, n * hv).view(n, hv, 1)).to(dtype)
    x[0, 0] = 0
    wide = (torch.randn(n, hv * dv + 24, generator=g) * 4).to(dtype)  # the gate as a column slice of a wider projection
    wide[0, :4] = torch.tensor([0.0, -200.0, 200.0, -88.0]).to(dtype)
    w = (1 + torch.randn(dv, generator=g) * 0.3).to(dtype)
    z = wide[:, :hv * dv]
    ref = gated_rms_norm(x.reshape(-1, dv), z.reshape(-1, dv), w, 1e-6).reshape(n, hv * dv).double()
    with torch.no_grad():
        y = _gated_norm(x.to(gpu), wide.to(gpu)[:, :hv * dv], w.to(gpu), 1e-6)
    torch.cuda.synchronize()
    y = y.cpu().double()
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    tiny = 1e-30 if dtype == torch.bfloat16 else 2.0 ** -24
    assert ((y - ref).abs() <= 3 * (ulp * ref.abs() + tiny)).all(), (y - ref).abs().max().item()
    assert (y == ref).double().mean().item() >= 0.999 or n * hv * dv < 1000


def test_gated_norm_special_values(gpu):
    """NaN and infinities come out where the eager ops give them."""
    x = torch.randn(6, 1, 64, generator=torch.Generator().manual_seed(1)).bfloat16()
    z = torch.randn(6, 64, generator=torch.Generator().manual_seed(2)).bfloat16()
    x[1, 0, 5], x[2, 0, 7], z[3, 3], z[4, 9], z[5, 1] = float("nan"), float("inf"), float("inf"), float("-inf"), float("nan")
    w = torch.ones(64, dtype=torch.bfloat16)
    ref = gated_rms_norm(x[:, 0], z, w, 1e-6)
    with torch.no_grad():
        y = _gated_norm(x.to(gpu), z.to(gpu), w.to(gpu), 1e-6).cpu()
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isinf(), ref.isinf())
    fine = ref.isfinite()
    assert ((y - ref)[fine].abs() <= 3 * 2.0 ** -7 * ref[fine].abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_of_every_gate(gpu, dtype):
    """Rows that normalize to 1 leave rnd(silu(gate)): every finite gate of the
    type down to -88.5 (where exp still fits fp32), within half a spacing of the value
    in 64 bits and 2^-20 of that value, which is what fp32 operations leave."""
    print(f"[gpu-case] silu of every gate, {dtype}", flush=True)
    z = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(dtype)
    z = z[z.isfinite() & (z >= -88.5)]
    z = torch.cat([z, z.new_zeros(-z.numel() % 64)]).view(-1, 64)
    x = torch.full((z.shape[0], 1, 64), 1024.0, dtype=dtype) if dtype == torch.bfloat16 else torch.full((z.shape[0], 1, 64), 64.0, dtype=dtype)
    with torch.no_grad():
        y = _gated_norm(x.to(gpu), z.to(gpu), torch.ones(64, dtype=dtype, device=gpu), 1e-6).cpu().double()
    ref = z.double() * torch.sigmoid(z.double())
    digits, least = (8, 2.0 ** -133) if dtype == torch.bfloat16 else (11, 2.0 ** -24)  # significant bits; the smallest value
    spacing = torch.ldexp(torch.ones_like(ref), torch.frexp(ref).exponent - digits).clamp(min=least)
    assert ((y - ref).abs() <= 0.5 * spacing + 2.0 ** -20 * ref.abs()).all()
