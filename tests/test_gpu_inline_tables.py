"""Prefix-cache tables and save tables that ride in a launch's arguments
(DanTreeAttnArgs.pasts_host, DanQkvFrontArgs.saves_host) against the uploaded
ones: up to 8 prefix entries and 16 saves go inline, one more is uploaded."""
import sys

import pytest
import torch

from dan_amd import _native
from dan_amd.attention import Batch, _attend_fused, _op_args, attend, segment, workspace_bytes
from dan_amd.front import qkv_front
from oracle import tree_attention as oracle

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def case(gpu, pasts, seed, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    segs, at = Batch(), 0
    for i in range(pasts):
        ids = [0] * (3 + 5 * i) + [1] * 4 + [2] * 2
        p = 9 + 31 * i
        past = {layer: tuple(torch.randn(2, p, 64, generator=g).to(dtype).to(gpu) for _ in range(2)) for layer in (0, 3)}
        segs.append(segment(at, ids, past, 0, p, str(gpu)))
        at += len(ids)
    q = torch.randn(at, 8, 64, generator=g).to(dtype).to(gpu).transpose(0, 1)
    k, v = (torch.randn(at, 2, 64, generator=g).to(dtype).to(gpu).transpose(0, 1) for _ in range(2))
    return q, k, v, segs


@pytest.mark.parametrize("pasts", [1, 8, 9])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_inline_prefix_table(gpu, pasts, dtype):
    say(f"{pasts} prefix entries, {dtype}")
    q, k, v, segs = case(gpu, pasts, pasts, dtype)
    outs = {layer: attend(q, k, v, segs, layer) for layer in (0, 3, 0)}
    torch.cuda.synchronize()
    assert (segs.tile_plan.past_hosts[0] is None) == (pasts > _native.INLINE_PASTS)
    for layer in (0, 3):
        ref = oracle.attend_dense(q, k, v, segs, layer)
        assert (outs[layer].float().cpu() - ref).abs().max().item() <= 2e-2
        fresh = Batch(segs)
        assert torch.equal(torch.ops.dan_amd.tree_attn(*_op_args(q, k, v, fresh, layer, None), None), outs[layer])  # uploaded
        assert torch.equal(attend(q, k, v, list(segs), layer), outs[layer])  # a plan of its own per call


def test_attention_only_launch_finds_its_table(gpu):
    """A PHASE_ATTEND call whose plan no copy has filled the table of (a plain
    list of segments: a new plan per call) uploads it."""
    say("attention-only launch on a fresh plan")
    q, k, v, segs = case(gpu, 3, 5)
    want = attend(q, k, v, segs, 0)
    ws = torch.empty(workspace_bytes(q, k, segs), dtype=torch.uint8, device=gpu)
    _attend_fused(q, k, v, segs, 0, None, phases=_native.PHASE_PACK, workspace=ws)
    out = _attend_fused(q, k, v, list(segs), 0, None, phases=_native.PHASE_ATTEND, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("first", [_native.PHASE_PACK, _native.PHASES_ALL])
def test_attention_only_launch_uses_the_filled_table(gpu, monkeypatch, first):
    """Behind a launch that filled the table (on its stream) an attention-only
    one uploads nothing; on another stream, or behind a captured launch that
    has not run, it does."""
    say(f"attention-only launches behind phases {first}")
    q, k, v, segs = case(gpu, 3, 6)
    want = attend(q, k, v, Batch(segs), 0)
    ws = torch.empty(workspace_bytes(q, k, segs), dtype=torch.uint8, device=gpu)
    pinned, pin = [], torch.Tensor.pin_memory
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t, *a: (pinned.append(t.numel()), pin(t, *a))[1])
    only = lambda: _attend_fused(q, k, v, segs, 0, None, phases=_native.PHASE_ATTEND, workspace=ws)  # noqa: E731
    _attend_fused(q, k, v, segs, 0, None, phases=first, workspace=ws)
    outs = [only(), only()]
    torch.cuda.synchronize()
    assert not pinned and all(torch.equal(o, want) for o in outs)
    side = torch.cuda.Stream(gpu)
    with torch.cuda.stream(side):
        out = only()
    torch.cuda.synchronize()
    assert len(pinned) == 1 and torch.equal(out, want)
    fresh = Batch(segs)
    workspace_bytes(q, k, fresh)  # plans outside the capture
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _attend_fused(q, k, v, fresh, 0, None, phases=first, workspace=ws)
    assert not fresh.tile_plan.past_filled


@pytest.mark.parametrize("saves", [1, 16, 17])
def test_inline_saves(gpu, saves):
    say(f"{saves} saves")
    g = torch.Generator().manual_seed(saves)
    segs, at = Batch(), 0
    for i in range(saves + 1):
        ids = [0] * (4 + i) + [1] * 3
        segs.append(segment(at, ids, None, 0 if i == 1 else 1 + i % 4, 0, str(gpu)))
        at += len(ids)
    qkv = torch.randn(at, 12, 64, generator=g).bfloat16().to(gpu)
    q, k, v = qkv.split((8, 2, 2), dim=1)
    ang = torch.randn(at, 64, generator=g)
    cos, sin = ang.cos().bfloat16().to(gpu), ang.sin().bfloat16().to(gpu)
    _, ko, vo = qkv_front(q, k, v, cos, sin, norm=None, segments=segs, layer=2)
    torch.cuda.synchronize()
    for s in segs:
        assert bool(s.saved) == bool(s.save)
        if s.save:
            assert torch.equal(s.saved[2][0], ko[:, s.start:s.start + s.save])
            assert torch.equal(s.saved[2][1], vo[:, s.start:s.start + s.save])


def test_graph_replays_with_inline_tables(gpu):
    """A captured call (front end with a save, attention with prefixes) replays with the table it was captured with."""
    say("graph replay with inline tables")
    q, k, v, segs = case(gpu, 2, 11)
    q, k, v = (t.clone() for t in (q, k, v))
    attend(q, k, v, segs, 0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attend(q, k, v, segs, 0)
        out3 = attend(q, k, v, segs, 3)  # a layer whose table is first made under capture
    for i in range(3):
        q.copy_(torch.randn(q.shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(i)))
        graph.replay()
        eager = attend(q, k, v, Batch(segs), 0), attend(q, k, v, Batch(segs), 3)
        torch.cuda.synchronize()
        assert torch.equal(out, eager[0]) and torch.equal(out3, eager[1])
