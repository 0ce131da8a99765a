"""Half tiles (each key tile split between the two halves of a work group's
waves) against the oracle and against whole tiles, at the sizes where the
split can go wrong: segments shorter than a wave, trunks that end inside the
first 32 keys (a half that sees no key of its first tile starts from its
partner's running max), tiles that hold past and new keys, ragged last tiles, GQA
ratios with 4, 2 and 1 heads per work group and with a second head chunk.

Bars: 2e-2 against the oracle as in tests/test_gpu_parity.py; against whole
tiles the halves add the same terms in another order, and P is rounded to
fp16 against another running max: 2^-9 of the largest |v| (two 2^-11
roundings of P, averaged weights) plus one spacing of the output type."""
import sys

import pytest
import torch

from dan_amd import _native
from dan_amd import attention as A
from dan_amd.workloads import build, to_e4m3
from oracle import tree_attention as oracle

import numpy as np

pytestmark = pytest.mark.gpu


def both(w, monkeypatch, **kw):
    lib = _native.load()
    h, n, d = w.q.shape
    outs = []
    for units in (10 ** 9, 0):  # never / always half tiles
        monkeypatch.setattr(A, "HALF_TILE_UNITS", units)
        w.segments.tile_plan = None
        outs.append(A.attend(w.q, w.k, w.v, w.segments, w.layer, **w.attend_kwargs, **kw))
        assert w.segments.tile_plan.tile_q == _native.tile_q(h, w.k.shape[0], d, lib=lib) // (1 if units else 2)
    torch.cuda.synchronize()
    return outs


SHAPES = [("short", [(1, [1]), (5, [3, 1, 40]), (31, [33]), (32, [1, 70])], [0, 0, 0, 0]),
          ("edges", [(64, []), (63, [2, 64]), (65, [31, 32, 33]), (200, [7] * 9)], [0, 0, 0, 0]),
          ("pasts", [(40, [5, 9, 1]), (7, [30]), (1, [3] * 6), (130, [17, 2])], [33, 64, 1, 200])]


@pytest.mark.parametrize("name,shape,pasts", SHAPES)
@pytest.mark.parametrize("heads", [(8, 2), (14, 2), (4, 2), (3, 3)])
@pytest.mark.parametrize("d,dtype", [(64, torch.float32), (64, torch.float16), (128, torch.bfloat16), (128, "e4m3"), (64, "e4m3")])
def test_half_tiles(gpu, monkeypatch, name, shape, pasts, heads, d, dtype):
    print(f"[gpu-case] half tiles {name} heads {heads} x {d} {dtype}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(d + heads[0])
    w = build(name, shape, heads[0], heads[1], d, torch.bfloat16 if dtype == "e4m3" else dtype, gpu, rng, per_segment_past=pasts)
    w = to_e4m3(w) if dtype == "e4m3" else w
    whole, half = both(w, monkeypatch)
    spacing = 2.0 ** -7 if half.dtype == torch.bfloat16 else 2.0 ** -10
    vmax = w.v.float().abs().max().item() * (w.meta["v_scale"].item() if dtype == "e4m3" else 1.0)
    assert (whole.float() - half.float()).abs().max().item() <= 2.0 ** -9 * vmax + spacing * whole.float().abs().max().item()
    if dtype != "e4m3":
        ref = oracle.attend_dense(w.q, w.k, w.v, w.segments, w.layer)
        assert (half.float().cpu() - ref).abs().max().item() <= 2e-2


def test_half_tiles_overflowing_units(gpu, monkeypatch):
    """Scores that grow along the trunk overflow fp16 P against the first
    tile's maximum: the unit runs again with the check, in both halves or in one."""
    print("[gpu-case] half tiles: growing scores", flush=True)
    rng = np.random.default_rng(5)
    w = build("grow", [(300, [20, 40])], 8, 2, 64, torch.float32, gpu, rng)
    n = w.num_tokens
    ramp = torch.linspace(0, 60, n, device=gpu)
    ramp[::3] *= -1
    for t in (w.q, w.k):
        t[..., 1:] *= 0.1
    w.q[..., 0] = 8.0
    w.k[..., 0] = ramp
    whole, half = both(w, monkeypatch)
    ref = oracle.attend_dense(w.q, w.k, w.v, w.segments, w.layer)
    for out in (whole, half):
        assert torch.isfinite(out).all()
        assert (out.float().cpu() - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("trunk,past", [(20, 0), (32, 0), (1, 31), (0, 8)])
@pytest.mark.parametrize("heads,d,dtype", [((32, 8), 128, torch.bfloat16), ((4, 4), 64, torch.bfloat16), ((8, 2), 128, "e4m3")])
def test_short_trunks_start_from_the_whole_first_tile(gpu, monkeypatch, trunk, past, heads, d, dtype):
    """Past and trunk within the first 32 keys: a branch whose keys begin in a
    later tile sees none of keys 32-63 of the first one. Both halves start from
    the tile's maximum (past and trunk score 30 powers of 2 above the branches, and
    their values are 0), so a branch key's p rounds to 0 in both, as in whole
    tiles. A half that ran again from its own keys' maximum would leave 2^-30."""
    print(f"[gpu-case] half tiles, past {past} trunk {trunk}, heads {heads} x {d} {dtype}", flush=True)
    rng = np.random.default_rng(trunk)
    w = build("short", [(trunk, [70, 60, 90])], heads[0], heads[1], d, torch.bfloat16, gpu, rng, per_segment_past=[past])
    for t in (w.q, w.k, w.v):
        t.zero_()
    top = 30 * 0.6931471805599453 * d ** 0.5 / 8
    w.q[..., 0] = 8
    w.k[:, :trunk, 0] = top
    w.v[:, trunk:] = 1
    if past:
        pk, pv = w.segments[0].past[0]
        pk.zero_()
        pk[..., 0] = top
        pv.zero_()
    w = to_e4m3(w) if dtype == "e4m3" else w
    whole, half = both(w, monkeypatch)
    branches = slice(trunk + 70, None)  # those whose keys begin past the first tile
    assert not whole[:, branches].any() and not half[:, branches].any()


def test_rule_of_one_segment(gpu):
    lib = _native.load()
    cus = A._num_cus(torch.device(gpu))
    tile = lambda h, hkv, d, n: A._tile_q(h, hkv, d, n, torch.device(gpu))  # noqa: E731
    if cus == 256:
        assert tile(32, 8, 128, 1024) == 32 and tile(32, 8, 128, 1025) == 64
        assert tile(8, 2, 64, 4096) == 32 and tile(8, 2, 64, 4097) == 64
    assert tile(16, 2, 256, 16) == _native.tile_q(16, 2, 256, lib=lib)
    assert tile(12, 8, 128, 16) == 0


@pytest.mark.parametrize("lens,want", [([40] * 25, 64), ([70] * 10, 32), ([20] * 50, 32)])
def test_segments_make_their_own_units(gpu, lens, want):
    """About 1000 tokens in many segments: half tiles only while all their units are resident at once."""
    w = build("many", [(x, []) for x in lens], 32, 8, 128, torch.bfloat16, gpu, np.random.default_rng(1))
    for _ in range(2):  # the second call finds the plan
        out = A.attend(w.q, w.k, w.v, w.segments, w.layer)
        if A._num_cus(torch.device(gpu)) == 256:
            assert w.segments.tile_plan.tile_q == want
    ref = oracle.attend_dense(w.q, w.k, w.v, w.segments, w.layer)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("planner", ["host", "device"])
def test_a_plan_made_ahead_is_kept(gpu, planner):
    """A small batch planned with whole tiles before layer 0 (get_plan) runs on that plan."""
    w = build("ahead", [(300, [20, 40])], 32, 8, 128, torch.bfloat16, gpu, np.random.default_rng(3))
    ref = A.attend(w.q, w.k, w.v, list(w.segments), w.layer)  # a plan of its own: half tiles
    plan = A.get_plan(w.segments, w.num_tokens, _native.tile_q(32, 8), gpu, planner=planner,
                      **(dict(groups=8, num_cus=A._num_cus(torch.device(gpu))) if planner == "device" else {}))
    out = A.attend(w.q, w.k, w.v, w.segments, w.layer)
    torch.cuda.synchronize()
    assert w.segments.tile_plan is plan
    assert (out.float() - ref.float()).abs().max().item() <= 2.0 ** -9 * w.v.float().abs().max().item() + 2.0 ** -7 * ref.float().abs().max().item()


@pytest.mark.parametrize("segments,want", [(1, 32), (4, 32), (16, 64)])
def test_budget_plan_counts_its_capacity(gpu, segments, want):
    """A BudgetPlan takes the form for the most units its capacities allow; its
    results are attend's, up to the rounding of P where that takes the other form."""
    w = build("budget", [(700, [60, 74])], 32, 8, 128, torch.bfloat16, gpu, np.random.default_rng(2))
    bp = A.BudgetPlan(w.num_tokens, 32, 8, 128, torch.bfloat16, gpu, max_segments=segments, max_branches=8)
    if A._num_cus(torch.device(gpu)) == 256:
        assert bp.tile_q == want
    bp.load(w.segments)
    got, out = bp.attend(w.q, w.k, w.v, w.layer).float(), A.attend(w.q, w.k, w.v, w.segments, w.layer).float()
    bar = 2.0 ** -9 * w.v.float().abs().max().item() + 2.0 ** -7 * out.abs().max().item() if want == 64 else 0.0
    assert (got - out).abs().max().item() <= bar


def test_half_tiles_need_their_flag():
    """A work item of half the queries is refused without key_halves = 2 (tests/test_abi.py), and the flag at head_dim 256."""
    from test_abi import _args
    import ctypes
    lib = _native.load()
    for kw in (dict(key_halves=2), dict(key_halves=3, tile_q=32), dict(key_halves=2, head_dim=256, tile_q=16)):
        assert lib.dan_tree_attn_fwd(ctypes.byref(_args(**kw)), None) == _native.ERR_INVALID_ARGUMENT
    assert lib.dan_tree_attn_fwd(ctypes.byref(_args(key_halves=2, tile_q=32)), None) == _native.OK  # no work: nothing runs
