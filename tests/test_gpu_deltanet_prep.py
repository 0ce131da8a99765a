"""The chunk preparation's block inverse of (I + L): runs that end inside, at and
past its 16-row blocks, with keys much alike and beta near 1 (T far from I),
against the recurrence in float64."""
import sys

import pytest
import torch

from dan_amd.deltanet import delta_rule

pytestmark = pytest.mark.gpu


def _recurrence(q, k, v, g, b, s):
    q, k, v, g, b, s = (x.double() for x in (q, k, v, g, b, s))
    q = q / (q.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt() * q.shape[-1] ** -0.5
    k = k / (k.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()
    out = []
    for t in range(q.shape[0]):
        s = s * g[t].exp()[:, None, None]
        u = (v[t] - (k[t][:, None] @ s)[:, 0]) * b[t][:, None]
        s = s + k[t][:, :, None] * u[:, None]
        out.append((q[t][:, None] @ s)[:, 0])
    return torch.stack(out), s


# The state's bar, of its largest value: fp32 arithmetic over at most 130 steps of
# about two roundings each (2^-24) for fp16 inputs; for bf16 the operands of the
# five products as pairs, two 2^-17 a product, on top.
@pytest.mark.parametrize("dtype,bar", [(torch.float16, 260 * 2.0 ** -24), (torch.bfloat16, 10 * 2.0 ** -17 + 260 * 2.0 ** -24)])
def test_alike_keys_at_block_edges(gpu, dtype, bar):
    gen = torch.Generator().manual_seed(21)
    lengths, h, dv = [1, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, 81, 130], 2, 32
    n = sum(lengths)
    q, v = torch.randn(n, h, 128, generator=gen).to(dtype), torch.randn(n, h, dv, generator=gen).to(dtype)
    k = (0.2 * torch.randn(n, h, 128, generator=gen) + torch.randn(1, h, 128, generator=gen)).to(dtype)
    g, b = -0.002 * torch.rand(n, h, generator=gen), 0.95 + 0.05 * torch.rand(n, h, generator=gen)
    st = 0.1 * torch.randn(len(lengths), h, 128, dv, generator=gen)
    print(f"[gpu-case] delta rule, alike keys {dtype} {lengths}", flush=True)
    sys.stdout.flush()
    o, f = delta_rule(*(x.to(gpu) for x in (q, k, v, g, b)), lengths, st.to(gpu), form="chunk")
    o, f = o.cpu().double(), f.cpu().double()
    eps = torch.finfo(dtype).eps
    at = 0
    for i, ln in enumerate(lengths):
        want, s = _recurrence(q[at:at + ln], k[at:at + ln], v[at:at + ln], g[at:at + ln], b[at:at + ln], st[i])
        assert (f[i] - s).abs().max() <= bar * s.abs().max(), (ln, float((f[i] - s).abs().max() / s.abs().max()))
        # an output is rounded to its type once; the sums' error is the state's
        got = o[at:at + ln]
        assert ((got - want).abs() <= 0.5 * eps * want.abs() + 2 * bar * want.abs().max() + 2.0 ** -24).all(), ln
        at += ln
