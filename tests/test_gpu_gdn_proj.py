"""dan_gdn_project (a DeltaNet layer's two narrow projections in one launch)
against float64, and the module calls it stands in for."""
import ctypes
import sys

import pytest
import torch
from torch import nn

from dan_amd import _native
from dan_amd.deltanet import NARROW_HIDDEN, _narrow_pair


def _case(n, cols, k, dtype, gpu, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, k, generator=g).to(dtype).to(gpu)
    lins = [nn.Linear(k, cols, bias=False, device=gpu, dtype=dtype) for _ in range(2)]
    for m in lins:
        m.weight.data.copy_((torch.randn(cols, k, generator=g) / k ** 0.5).to(dtype))
    return x, lins


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,cols,k", [(1, 4, 32), (15, 16, 64), (16, 20, 96), (17, 48, 2048), (834, 16, 2048), (33, 64, 2080),
                                      (5, 12, 544), (4097, 16, 64), (2050, 20, 160)])
def test_both_outputs(gpu, n, cols, k, dtype):
    print(f"[gpu-case] narrow projections {n} x {k} to 2 x {cols} {dtype}", flush=True)
    sys.stdout.flush()
    x, (m0, m1) = _case(n, cols, k, dtype, gpu)
    with torch.no_grad():
        got = _narrow_pair(x, m0, m1)
        padded = torch.zeros(n, k + 8, dtype=dtype, device=gpu)[:, :k].copy_(x)  # rows further apart: the same bits
        again = _narrow_pair(padded, m0, m1)
    torch.cuda.synchronize()
    for y, y2, m in zip(got, again, (m0, m1)):
        xd, w = x.cpu().double(), m.weight.detach().cpu().double()
        want, size = xd @ w.T, xd.abs() @ w.abs().T
        # k products in fp32, one rounding to the output's type
        bar = k * 2.0 ** -24 * size + 0.5 * torch.finfo(dtype).eps * want.abs() + torch.finfo(dtype).tiny
        assert y.dtype == dtype and y.is_contiguous() and torch.equal(y, y2)
        assert ((y.cpu().double() - want).abs() <= bar).all()


@pytest.mark.gpu
def test_other_modules_are_called_themselves(gpu):
    x, (m0, m1) = _case(9, 16, 64, torch.bfloat16, gpu)
    calls = []

    class Own(nn.Linear):
        def forward(self, x):
            calls.append("own")
            return super().forward(x)

    own = Own(64, 16, bias=False, device=gpu, dtype=torch.bfloat16)
    biased = nn.Linear(64, 16, bias=True, device=gpu, dtype=torch.bfloat16)
    many = nn.Linear(64, 16 * 257, bias=False, device=gpu, dtype=torch.bfloat16)  # more work groups than CUs
    with torch.no_grad():
        for a, b in ((own, m1), (biased, m1), (many, many)):
            y0, y1 = _narrow_pair(x, a, b)
            assert torch.equal(y0, a(x)) and torch.equal(y1, b(x))
        assert calls
        hook = m0.register_forward_hook(lambda m, i, o: o * 0)
        assert not _narrow_pair(x, m0, m1)[0].any()
        hook.remove()
        odd = torch.zeros(9, 65, dtype=torch.bfloat16, device=gpu)[:, 1:].copy_(x)  # misaligned rows
        assert torch.equal(_narrow_pair(odd, m0, m1)[0], m0(odd))
        deep = nn.Linear(NARROW_HIDDEN + 32, 16, bias=False, device=gpu, dtype=torch.bfloat16)
        xd = x.repeat(1, NARROW_HIDDEN // 64 + 1)[:, :NARROW_HIDDEN + 32]
        assert torch.equal(_narrow_pair(xd, deep, deep)[0], deep(xd))
        none = _narrow_pair(x[:0], m0, m1)
        assert none[0].shape == none[1].shape == (0, 16)
    y0, _ = _narrow_pair(x, m0, m1)  # gradients wanted
    assert y0.requires_grad


@pytest.mark.parametrize("kw,status,needle", [
    (dict(abi_version=1), _native.ERR_VERSION, "abi_version"), (dict(dtype=_native.DTYPE_F32), _native.ERR_UNSUPPORTED, "dtype"),
    (dict(cols=6), _native.ERR_UNSUPPORTED, "cols"), (dict(hidden=48), _native.ERR_UNSUPPORTED, "hidden"),
    (dict(x_stride=60), _native.ERR_INVALID_ARGUMENT, "strides"), (dict(y1_stride=18), _native.ERR_INVALID_ARGUMENT, "strides"),
    (dict(w0=4104), _native.ERR_INVALID_ARGUMENT, "aligned"), (dict(y0=4100), _native.ERR_INVALID_ARGUMENT, "aligned"),
    (dict(w1=None), _native.ERR_INVALID_ARGUMENT, "NULL"), (dict(rows=-1), _native.ERR_INVALID_ARGUMENT, "rows"),
    (dict(rows=0, x=None), _native.OK, "")])
def test_argument_errors(kw, status, needle):
    lib = _native.load()
    base = dict(abi_version=_native.GDN_ABI_VERSION, dtype=_native.DTYPE_BF16, rows=3, cols=16, hidden=64, x=4096, w0=4096, w1=4096,
                y0=4096, y1=4096, x_stride=64, w0_stride=64, w1_stride=64, y0_stride=16, y1_stride=16)
    a = _native.DanGdnProjArgs(**{**base, **kw})
    assert lib.dan_gdn_project(ctypes.byref(a), None) == status
    assert needle in _native.last_error(lib)
