"""The delta rule writing its runs' outputs to given rows (DanGdnArgs.out_start)
and its final states to a given buffer, and the conv phase reading A_log and
dt_bias in the model dtype: bit-identical to the plain calls."""
import sys
from types import SimpleNamespace

import pytest
import torch

from dan_amd.deltanet import _delta_rule, conv_phase, delta_rule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,dtype,lengths", [
    ("token", torch.bfloat16, [5, 0, 1, 70]), ("chunk", torch.bfloat16, [70, 5, 0, 130, 33, 64]),
    ("chunk", torch.float16, [300, 700, 1]), ("chunk", torch.float16, [70, 5, 0, 130, 33])])
def test_out_rows_equal_index_copy(gpu, form, dtype, lengths):
    print(f"[gpu-case] delta rule {form} {dtype} {lengths}: outputs to packed rows", flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(3)
    n, hk, hv, dv, r = sum(lengths), 2, 4, 64, len(lengths)
    q, k = (torch.randn(n, hk, 128, generator=g).to(dtype).to(gpu) for _ in range(2))
    v = torch.randn(n, hv, dv, generator=g).to(dtype).to(gpu)
    gate, beta = (-torch.rand(n, hv, generator=g) * 0.2).to(gpu), torch.rand(n, hv, generator=g).to(gpu)
    st = (torch.randn(r, hv, 128, dv, generator=g) * 0.1).to(gpu)
    o, f = delta_rule(q, k, v, gate, beta, lengths, st, form=form)
    rows = n + 40  # runs in reverse order of rows, with a gap of 7 before the last one placed
    start, at = [0] * r, 3
    for i in reversed(range(r)):
        start[i] = at
        at += lengths[i] + (7 if i == 1 else 0)
    start_d = torch.tensor(start, dtype=torch.int32, device=gpu)
    out = torch.full((rows, hv, dv), 5.0, dtype=dtype, device=gpu)
    fin = torch.empty(r + 2, hv, 128, dv, device=gpu)
    _delta_rule(q, k, v, gate, beta, lengths, st, form=form, out=out, out_start=start_d, finals=fin[2:])
    torch.cuda.synchronize()
    want = torch.full_like(out, 5.0)
    for i, ln in enumerate(lengths):
        want[start[i]:start[i] + ln] = o[sum(lengths[:i]):sum(lengths[:i]) + ln]
    assert torch.equal(out, want) and torch.equal(fin[2:], f)
    # starts outside the rows are clamped so that the run stays inside
    big = torch.tensor([10 ** 9] * r, dtype=torch.int32, device=gpu)
    out2 = torch.zeros(rows, hv, dv, dtype=dtype, device=gpu)
    _delta_rule(q[:lengths[0]], k[:lengths[0]], v[:lengths[0]], gate[:lengths[0]], beta[:lengths[0]], lengths[:1], st[:1], form=form,
                out=out2, out_start=big[:1])
    torch.cuda.synchronize()
    assert torch.equal(out2[rows - lengths[0]:], o[:lengths[0]])


def test_out_of_another_type_is_refused(gpu):
    z = torch.zeros(4, 2, 128, dtype=torch.bfloat16, device=gpu)
    args = (z, z, z, torch.zeros(4, 2, device=gpu), torch.zeros(4, 2, device=gpu), [4], torch.zeros(1, 2, 128, 128, device=gpu))
    with pytest.raises(ValueError, match="out"):
        _delta_rule(*args, out=torch.zeros(4, 2, 128, device=gpu), out_start=torch.zeros(1, dtype=torch.int32, device=gpu))
    with pytest.raises(RuntimeError, match="num_out_rows"):
        _delta_rule(*args, out=z[:3], out_start=torch.zeros(1, dtype=torch.int32, device=gpu))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_parameters_in_the_model_dtype(gpu, dtype):
    g = torch.Generator().manual_seed(4)
    n, c, hv = 37, 64, 3
    ph = SimpleNamespace(rows=torch.arange(n, dtype=torch.int32, device=gpu), ext=torch.arange(n + 3, dtype=torch.int32, device=gpu) - 3,
                         take=torch.arange(n, dtype=torch.int32, device=gpu))
    x, w = torch.randn(n, c, generator=g).to(dtype).to(gpu), torch.randn(c, 1, 4, generator=g).to(dtype).to(gpu)
    b, a = (torch.randn(n, hv, generator=g).to(dtype).to(gpu) for _ in range(2))
    al, dt = (torch.randn(hv, generator=g).to(dtype).to(gpu) for _ in range(2))
    one, two = conv_phase(x, None, ph, w, b, a, al, dt), conv_phase(x, None, ph, w, b, a, al.float(), dt.float())
    mixed = conv_phase(x, None, ph, w, b, a, al.float(), dt)
    torch.cuda.synchronize()
    for p, q, r in zip(one, two, mixed):
        assert torch.equal(p, q) and torch.equal(p, r)
