"""The planner's dealing and its moves and swaps, slot by slot against the same
rule in Python: few and many slots per head group, fewer items than a wave and
more than a work group, and loads of 2^24 key tiles and more."""
import sys

import numpy as np
import pytest
import torch

from dan_amd import plan as P
from dan_amd.attention import Batch, segment

pytestmark = pytest.mark.gpu


def _slots(cost, k, overhead=1):
    w = [int(c) + overhead for c in cost]
    load, slot = [0] * k, []
    for x in w:
        j = min(range(k), key=lambda j: (load[j], j))
        load[j] += x
        slot.append(j)
    for _ in range(2 * len(w) + 64):
        top = max(load)
        a = load.index(top)
        options = []
        for i in (i for i, s in enumerate(slot) if s == a):
            options += [(max(top - w[i], load[b] + w[i]), i, 0, b) for b in range(k) if b != a]
            options += [(max(top - d, load[slot[j]] + d), i, 1, j) for j, d in ((j, w[i] - w[j]) for j in range(len(w)))
                        if slot[j] != a and d > 0]
        best = min(options, default=(top,))
        if best[0] >= top:
            break
        _, i, swap, x = best
        b, d = (slot[x], w[i] - w[x]) if swap else (x, w[i])
        load[a] -= d
        load[b] += d
        slot[i] = b
        if swap:
            slot[x] = a
    return slot


# (trunk and branch lengths of the segments, past lengths, queries a tile, head groups, CUs)
CASES = {
    "fewer items than a wave": (((700, (30, 60)), (90, (16,) * 5)), (0, 300), 64, 4, 24),
    "more slots than lanes": (tuple((97 + 61 * i, (9 + i, 40)) for i in range(9)), (0,) * 9, 16, 1, 256),
    "more items than threads": (tuple((1501 + 137 * i, (50, 77)) for i in range(8)), (640,) * 8, 16, 4, 160),
    "loads past 24 bits": (tuple((201 + 97 * i, (33,)) for i in range(5)), tuple((1 << 26) + 4096 * i for i in range(5)), 32, 2, 26),
}


@pytest.mark.parametrize("name", CASES)
def test_slots_follow_the_rule(gpu, name):
    structure, pasts, tile_q, groups, cus = CASES[name]
    segs, start = Batch(), 0
    for (trunk, lens), past in zip(structure, pasts):
        ids = [0] * trunk + [j for j, n in enumerate(lens, 1) for _ in range(n)]
        segs.append(segment(start, ids, None, 0, 0, "cuda"))
        segs[-1].past, segs[-1].past_len = ({0: None} if past else None), past
        start += len(ids)
    print(f"[gpu-case] planner rounds: {name}", flush=True)
    sys.stdout.flush()
    plan = P.TilePlan.build_device(segs, start, tile_q, gpu, groups, cus)
    torch.cuda.synchronize()
    cost, work = plan.cost_d.cpu().numpy()[:plan.num_work], plan.work_d.cpu().numpy()[:plan.num_work]
    units, off, slots = plan.schedules[(groups, cus)]
    units, off = units.cpu().numpy(), off.cpu().numpy()
    want = _slots(cost, slots // groups)
    rank = {tuple(r): i for i, r in enumerate(work)}
    for s in range(slots):
        got = [rank[tuple(u[:8])] for u in units[off[s]:off[s + 1]]]
        assert got == [i for i, j in enumerate(want) if j == s // groups], (name, s)
    if name == "loads past 24 bits":
        assert (int(cost[0]) + 1) * len(cost) >= 1 << 24
