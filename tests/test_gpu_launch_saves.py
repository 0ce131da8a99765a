"""attend's prefix saves written by the V^T copy's launch: the clones' values,
shapes and strides, for every layout that takes the launch and those that do not."""
import ctypes
import sys

import pytest
import torch

from dan_amd import _native
from dan_amd.attention import Batch, Segment, _launch_saves, attend, segment


def _batch(lengths, saves):
    segs, start = Batch(), 0
    for n, save in zip(lengths, saves):
        ids = [0] * (n - n // 4) + [1] * (n // 4)
        segs.append(segment(start, ids, None, save, 0, "cuda"))
        start += n
    return segs, start


def _qkv(layout, h, hkv, n, d, dtype, gpu):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(n, h + 2 * hkv, d, generator=g).to(dtype).to(gpu)
    q, k, v = x[:, :h].transpose(0, 1), x[:, h:h + hkv].transpose(0, 1), x[:, h + hkv:].transpose(0, 1)
    if layout == "heads":
        k, v = k.contiguous(), v.contiguous()
    elif layout == "mixed":  # clones keep the order of the dimensions
        k, v = k.contiguous(), v
    elif layout == "tokens":
        k, v = (t.transpose(0, 1).contiguous().transpose(0, 1) for t in (k, v))
    elif layout == "misaligned":
        k, v = (torch.zeros(hkv, n, d + 1, dtype=dtype, device=gpu)[:, :, 1:].copy_(t) for t in (k, v))
    return q, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["fused", "heads", "tokens", "mixed", "misaligned"])
@pytest.mark.parametrize("lengths,saves,d,dtype", [([5], [1], 64, torch.bfloat16), ([130, 9, 300], [97, 0, 225], 128, torch.float16),
                                                   ([64], [48], 256, torch.bfloat16), ([20] * 9, [3] * 9, 64, torch.bfloat16),
                                                   ([33] * 8, [2, 3, 4, 5, 6, 7, 8, 25], 128, torch.bfloat16), ([9], [2], 128, torch.bfloat16)])
def test_saves_equal_clones(gpu, layout, lengths, saves, d, dtype):
    segs, n = _batch(lengths, saves)
    q, k, v = _qkv(layout, 4, 2, n, d, dtype, gpu)
    print(f"[gpu-case] saves {saves} of {lengths} d {d} {dtype} {layout}", flush=True)
    sys.stdout.flush()
    with torch.no_grad():
        out = attend(q, k, v, segs, 3)
        plain = attend(q, k, v, segs, 3, save=False)
    torch.cuda.synchronize()
    assert torch.equal(out, plain)
    assert bool(_launch_saves(k, v, segs)) == (len(saves) <= 8 and saves != [1])
    for s in segs:
        if s.save:
            for got, t in zip(s.saved[3], (k, v)):
                want = t[:, s.start:s.start + s.save].clone()
                assert torch.equal(got, want) and got.stride() == want.stride()
        else:
            assert not s.saved


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["heads expanded", "one expanded", "tokens expanded", "columns outermost", "columns strided", "heads innermost"])
def test_saves_of_other_layouts_equal_clones(gpu, layout):
    """Values and strides of the clones where a stride is 0 or head_dim is not the innermost dimension."""
    print(f"[gpu-case] saves, {layout}", flush=True)
    segs, n = _batch([40, 30], [17, 9])
    q, k, v = _qkv("heads", 4, 2, n, 64, torch.bfloat16, gpu)
    if layout == "heads expanded":
        k, v = k[:1].expand(2, n, 64), v[:1].expand(2, n, 64)
    elif layout == "one expanded":
        v = v[:1].expand(2, n, 64)
    elif layout == "tokens expanded":
        k = k[:, :1].expand(2, n, 64)
    elif layout == "columns outermost":
        k, v = (t.permute(2, 0, 1).contiguous().permute(1, 2, 0) for t in (k, v))
    elif layout == "columns strided":
        k, v = (torch.zeros(2, n, 128, dtype=t.dtype, device=gpu)[:, :, ::2].copy_(t) for t in (k, v))
    else:
        k, v = (t.permute(1, 2, 0).contiguous().permute(2, 0, 1) for t in (k, v))
    with torch.no_grad():
        out = attend(q, k, v, segs, 3)
        plain = attend(q, k.contiguous(), v.contiguous(), segs, 3, save=False)
    torch.cuda.synchronize()
    assert torch.equal(out, plain)
    for s in segs:
        for got, t in zip(s.saved[3], (k, v)):
            want = t[:, s.start:s.start + s.save].clone()
            assert torch.equal(got, want) and got.stride() == want.stride()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_batch_reads_what_it_saves(gpu, dtype):
    """A request whose prefix is the rows that another of its batch saves: each
    layer's entry is there before the plan and the launch read it."""
    print(f"[gpu-case] a save read in its own batch, {dtype}", flush=True)
    first = segment(0, [0] * 50 + [1] * 7, None, 31, 0, "cuda")
    second = Segment(57, 80, 13, [(70, 80)], first.saved, past_len=31, branch_ids=[0] * 13 + [1] * 10, device="cuda")
    segs = Batch([first, second])
    with torch.no_grad():
        for layer in (0, 1):
            q, k, v = (t + layer for t in _qkv("fused", 4, 2, 80, 64, dtype, gpu))
            out = attend(q, k, v, segs, layer)
            entry = {layer: (k[:, :31].clone(), v[:, :31].clone())}
            apart = Batch([segment(0, first.branch_ids, None, 0, 0, "cuda"), segment(57, second.branch_ids, entry, 0, 31, "cuda")])
            assert torch.equal(out, attend(q, k, v, apart, layer))
            assert all(torch.equal(a, b) for a, b in zip(first.saved[layer], entry[layer]))


@pytest.mark.gpu
def test_rows_past_the_segment_are_cloned(gpu):
    segs, n = _batch([20, 30], [0, 0])
    segs[0].save = 25  # into the next segment, as a clone allows
    q, k, v = _qkv("fused", 4, 2, n, 64, torch.bfloat16, gpu)
    assert not _launch_saves(k, v, segs)


@pytest.mark.parametrize("kw,needle", [(dict(num_saves=9), "num_saves"), (dict(num_saves=-1), "num_saves"), (dict(save_layout=4), "save_layout"), (dict(saves=None), "num_saves"), (dict(num_work=0), "num_saves"),
                                       (dict(in_dtype=_native.DTYPE_E4M3, v_dtype=_native.DTYPE_E4M3, q_scale=4096, k_scale=4096, v_scale=4096), "num_saves"),
                                       (dict(start=90), "save 0"), (dict(len=0), "save 0"), (dict(k_dst=4104), "aligned")])
def test_argument_errors(kw, needle):
    lib = _native.load()
    entry = dict(start=0, len=20, k_dst=4096, v_dst=4096)
    entry.update({k: kw[k] for k in entry if k in kw})
    table = (_native.DanTreeAttnSave * 1)(tuple(entry.values()))
    base = dict(abi_version=_native.ABI_VERSION, in_dtype=_native.DTYPE_BF16, out_dtype=_native.DTYPE_BF16, v_dtype=_native.DTYPE_BF16,
                num_heads=4, num_kv_heads=2, head_dim=128, num_tokens=100, scale=1.0, q=4096, k=4096, v=4096, out=4096, segments=4096,
                num_segments=1, work=4096, num_work=1, key_lo=4096, tile_q=_native.tile_q(4, 2), vt_cols=128, col_seg=4096,
                num_saves=1, saves=ctypes.addressof(table))
    a = _native.DanTreeAttnArgs(**{**base, **{k: x for k, x in kw.items() if k not in entry}})
    assert lib.dan_tree_attn_fwd(ctypes.byref(a), None) == _native.ERR_INVALID_ARGUMENT
    assert needle in _native.last_error(lib)
    if "num_work" in kw:
        assert lib.dan_tree_attn_fwd_noalloc(ctypes.byref(a), None) == _native.ERR_INVALID_ARGUMENT
