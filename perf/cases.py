"""The calls that a program built on this package makes, as measurable cases.

Four kinds, each through public entry points:

- ``attend``: one attention layer's call over a packed tree batch
  (``dan_amd.attention.attend``), the batch's plan kept as a forward keeps it
  for its layers;
- ``forward``: the attention side of a whole prefill forward: a new ``Batch``
  (so the tile plan is made), then per layer the front end (``qkv_front``:
  q/k norm, rotary, prefix save) and ``attend``;
- ``fp8``: one e4m3 decoder linear (``dan_amd.quant.FP8Linear``): the
  per-call quantization of the activations and the scaled GEMM;
- ``deltanet``: one Gated DeltaNet layer (``dan_amd.deltanet.DeltaNet``) over
  a packed tree batch with cached prefixes and a save boundary.

Batches are trees as the serving engine packs them: requests of one trunk (the
prompt) and several branches (the questions), packed in order up to a token
budget of 8192. Structures come from a case's ``tree`` seed, values from the
seed given to ``prepare``.
"""
import math
import random
from types import SimpleNamespace

import torch

from dan_amd.attention import Batch, attend, segment
from dan_amd.deltanet import DeltaNet
from dan_amd.front import qkv_front
from dan_amd.quant import FP8Linear
from dan_amd.workloads import branch_ids, fifo_pack, quantize_e4m3

BUDGET = 8192
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "e4m3": torch.bfloat16}
LLAMA3_8B = dict(heads=32, kv_heads=8, head_dim=128)
LLAMA3_8B_LINEARS = ((6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336))  # qkv, o, gate_up, down: (N, K)


def _tree_fields(tree, requests, trunk, branches, length, budget=BUDGET):
    return dict(tree=tree, requests=requests, trunk_lo=trunk[0], trunk_hi=trunk[1], branches_lo=branches[0],
                branches_hi=branches[1], length_lo=length[0], length_hi=length[1], budget=budget)


def listed():
    return [
        # The smallest call: one short request in fp32, where launches and host time count.
        dict(name="attend_fp32_small", kind="attend", dtype="fp32", heads=8, kv_heads=2, head_dim=64, past=0, save=False,
             **_tree_fields(1, 1, (256, 256), (4, 4), (32, 32))),
        # One interactive request of a few hundred tokens on the 8B shape, its prompt's prefix kept for later reads.
        dict(name="attend_bf16_request", kind="attend", dtype="bf16", past=0, save=True, **LLAMA3_8B,
             **_tree_fields(2, 1, (641, 641), (5, 5), (9, 77))),
        # The serving budget: requests behind a shared cached prefix, packed to 8192 tokens.
        dict(name="attend_bf16_budget", kind="attend", dtype="bf16", past=1024, save=False, **LLAMA3_8B,
             **_tree_fields(3, 16, (200, 2000), (3, 12), (16, 96))),
        # One long document read with 32 short questions: the largest attention call.
        dict(name="attend_bf16_document", kind="attend", dtype="bf16", past=0, save=False, **LLAMA3_8B,
             **_tree_fields(4, 1, (7680, 7680), (32, 32), (16, 16))),
        # The serving budget with e4m3 q, k, v and prefix entries.
        dict(name="attend_e4m3_budget", kind="attend", dtype="e4m3", past=1024, save=False, **LLAMA3_8B,
             **_tree_fields(5, 16, (200, 2000), (3, 12), (16, 96))),
        # The hybrid models' gated-attention layout (head_dim 256) at the serving budget.
        dict(name="attend_d256_budget", kind="attend", dtype="bf16", heads=16, kv_heads=2, head_dim=256, past=1024,
             save=False, **_tree_fields(6, 16, (200, 2000), (3, 12), (16, 96))),
        # A prefill forward over four mid-sized requests: plan, front ends and attention of 16 layers.
        dict(name="forward_reads", kind="forward", dtype="bf16", layers=16, norm="rms", rotary=128, past=300, save=True,
             **LLAMA3_8B, **_tree_fields(7, 4, (128, 1024), (3, 6), (16, 64))),
        # FP8 linears: the output projection for one short request,
        dict(name="fp8_o_short", kind="fp8", dtype="bf16", tokens=77, n=4096, k=4096, rowwise=True, bias=False),
        # the down projection for a few requests,
        dict(name="fp8_down_requests", kind="fp8", dtype="bf16", tokens=1037, n=4096, k=14336, rowwise=True, bias=False),
        # and the gate/up projection at the full budget.
        dict(name="fp8_gate_up_budget", kind="fp8", dtype="bf16", tokens=8192, n=28672, k=4096, rowwise=True, bias=False),
        # A DeltaNet layer for one request, and at the full budget behind cached prefixes.
        dict(name="deltanet_request", kind="deltanet", dtype="bf16", hidden=2048, k_heads=16, v_heads=16, v_dim=128,
             past=False, save=True, **_tree_fields(8, 1, (611, 611), (5, 5), (9, 77))),
        dict(name="deltanet_budget", kind="deltanet", dtype="bf16", hidden=2048, k_heads=16, v_heads=16, v_dim=128,
             past=True, save=True, **_tree_fields(9, 16, (200, 2000), (3, 12), (16, 96))),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_tree(rng, most):
    """Requests of about equal share of a log-uniform token count; trunks from a fifth to all but the branches."""
    total = _log(rng, 64, most)
    requests = rng.choice((1, 1, 2, 4, 8)) if total >= 512 else 1
    share = max(48, total // requests)
    nb = rng.randint(1, 8)
    length = (1, max(2, min(96, share // (2 * nb))))
    trunk = max(2, share - nb * (length[0] + length[1]) // 2)
    return _tree_fields(rng.randrange(1 << 30), requests, (max(1, trunk // 2), trunk), (max(1, nb - 2), nb), length)


def draw(rng):
    kind = rng.choice(("attend", "attend", "forward", "fp8", "fp8", "deltanet"))
    if kind == "attend":
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32", "e4m3"))
        h, hkv, d = rng.choice(((32, 8, 128), (32, 8, 128), (16, 2, 256), (8, 2, 64), (32, 32, 128)))
        return dict(kind=kind, dtype=dtype, heads=h, kv_heads=hkv, head_dim=d, past=rng.choice((0, 0, _log(rng, 16, 2048))),
                    save=dtype != "e4m3" and rng.random() < 0.5, **_draw_tree(rng, 4096 if dtype == "fp32" else BUDGET))
    if kind == "forward":
        h, hkv, d = rng.choice(((32, 8, 128), (16, 2, 256)))
        return dict(kind=kind, dtype=rng.choice(("bf16", "fp16")), layers=rng.randint(2, 8),
                    norm=rng.choice(("none", "rms", "zero_centered")), rotary=rng.choice((64, d)), heads=h, kv_heads=hkv,
                    head_dim=d, past=rng.choice((0, _log(rng, 16, 512))), save=rng.random() < 0.5, **_draw_tree(rng, 3072))
    if kind == "fp8":
        n, k = rng.choice(LLAMA3_8B_LINEARS + ((16 * rng.randint(16, 512), 16 * rng.randint(16, 512)),))
        return dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "fp16")), tokens=_log(rng, 1, BUDGET), n=n, k=k,
                    rowwise=rng.random() < 0.8, bias=rng.random() < 0.3)
    hk, hv, dv = rng.choice(((16, 16, 128), (16, 32, 128), (16, 16, 64)))
    return dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "fp16")), hidden=rng.choice((1024, 2048)), k_heads=hk,
                v_heads=hv, v_dim=dv, past=rng.random() < 0.5, save=rng.random() < 0.5, **_draw_tree(rng, BUDGET))


def _structure(case):
    """[(trunk, [branch lengths])] of the case's requests, packed in order into its budget."""
    r = random.Random(case["tree"])
    reqs = []
    for _ in range(case["requests"]):
        trunk = r.randint(case["trunk_lo"], case["trunk_hi"])
        reqs.append((trunk, [r.randint(case["length_lo"], case["length_hi"])
                             for _ in range(r.randint(case["branches_lo"], case["branches_hi"]))]))
    return fifo_pack(reqs, case["budget"])[0]


def _tokens(case):
    return sum(t + sum(ls) for t, ls in _structure(case))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _saving(case, i, requests):
    """The last request keeps its prompt's prefix (the others start from the cache, where there is one)."""
    return case["save"] and i == requests - 1


# ------------------------------------------------------------------ inputs, from the seed alone


def _attend_inputs(case, seed):
    """The fused projection's rows [N, H + 2 Hkv, D] (after norm and rotary, of
    the size these have) and the shared prefix entry's k, v."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
    fused = _randn(g, _tokens(case), h + 2 * hkv, d, std=0.7, dtype=dt)
    q, k, v = (x.transpose(0, 1) for x in fused.split((h, hkv, hkv), dim=1))
    past = tuple(_randn(g, hkv, case["past"], d, std=0.7, dtype=dt) for _ in range(2)) if case["past"] else None
    return q, k, v, past


def _forward_inputs(case, seed):
    """Per layer the qkv projection's output, the prefix entry and the norm weights; the rotary tables."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    h, hkv, d, n, r = case["heads"], case["kv_heads"], case["head_dim"], _tokens(case), case["rotary"]
    pos = []
    for trunk, lens in _structure(case):
        pos += list(range(case["past"], case["past"] + trunk))
        for length in lens:
            pos += list(range(case["past"] + trunk, case["past"] + trunk + length))
    freq = 10000.0 ** (-torch.arange(0, r, 2, dtype=torch.float64) / r)
    ang = torch.tensor(pos, dtype=torch.float64)[:, None] * freq[None]
    ang = torch.cat([ang, ang], dim=1).cuda()
    layers = []
    for _ in range(case["layers"]):
        past = tuple(_randn(g, hkv, case["past"], d, std=0.7, dtype=dt) for _ in range(2)) if case["past"] else None
        base = 0.0 if case["norm"] == "zero_centered" else 1.0
        layers.append(SimpleNamespace(qkv=_randn(g, n, (h + 2 * hkv) * d, std=0.7, dtype=dt), past=past,
                                      qw=(base + _randn(g, d, std=0.1)).to(dt), kw=(base + _randn(g, d, std=0.1)).to(dt)))
    return layers, ang.cos().to(dt), ang.sin().to(dt)


def _fp8_inputs(case, seed):
    """Activations as a norm leaves them, a few channels large; weights of the usual spread."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    x = _randn(g, case["tokens"], case["k"])
    x[:, :: 97] *= 6.0
    w = _randn(g, case["n"], case["k"], std=0.02, dtype=dt)
    return x.to(dt), w, _randn(g, case["n"], std=0.1, dtype=dt) if case["bias"] else None


def _deltanet_inputs(case, seed):
    """The layer's parameters by name, its input rows and the cached (conv history, state) of every request but a saving one."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    hidden, hk, hv, dv, kernel = case["hidden"], case["k_heads"], case["v_heads"], case["v_dim"], 4
    conv = 2 * hk * 128 + hv * dv
    p = {"in_proj_qkv.weight": _randn(g, conv, hidden, std=hidden ** -0.5, dtype=dt),
         "in_proj_z.weight": _randn(g, hv * dv, hidden, std=hidden ** -0.5, dtype=dt),
         "in_proj_b.weight": _randn(g, hv, hidden, std=hidden ** -0.5, dtype=dt),
         "in_proj_a.weight": _randn(g, hv, hidden, std=hidden ** -0.5, dtype=dt),
         "conv1d.weight": _randn(g, conv, 1, kernel, std=0.5, dtype=dt),
         "dt_bias": (_randn(g, hv, std=0.5) - 3.0).to(dt), "A_log": _randn(g, hv, std=0.5).to(dt),
         "norm.weight": (1.0 + _randn(g, dv, std=0.1)).to(dt),
         "out_proj.weight": _randn(g, hidden, hv * dv, std=(hv * dv) ** -0.5, dtype=dt)}
    x = _randn(g, _tokens(case), hidden, dtype=dt)
    pasts, reqs = [], _structure(case)
    for i in range(len(reqs)):
        if case["past"] and not _saving(case, i, len(reqs)):
            pasts.append((_randn(g, kernel - 1, conv, dtype=dt), _randn(g, hv, 128, dv, std=0.05)))
        else:
            pasts.append(None)
    return p, x, pasts


# ------------------------------------------------------------------ what a program has in hand, and one pass


def _batch(case, past_of=lambda i: None, past_len=0):
    """The packed requests as a ``Batch``: request i starts from ``past_of(i)``."""
    segs, start, reqs = Batch(), 0, _structure(case)
    for i, (trunk, lens) in enumerate(reqs):
        ids = branch_ids(trunk, lens)
        save = max(1, trunk // 2) if _saving(case, i, len(reqs)) else 0
        segs.append(segment(start, ids, past_of(i), save, past_len, "cuda"))
        start += len(ids)
    return segs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attend":
        q, k, v, past = _attend_inputs(case, seed)
        scales, entry = {}, past
        if case["dtype"] == "e4m3":
            (q, qs), (k, ks), (v, vs) = quantize_e4m3(q), quantize_e4m3(k), quantize_e4m3(v)
            scales = dict(q_scale=qs, k_scale=ks, v_scale=vs)
            if past:
                (pk, pks), (pv, pvs) = quantize_e4m3(past[0]), quantize_e4m3(past[1])
                entry = (pk, pv, pks, pvs)
        shared = {0: entry} if past else None
        return dict(case=case, q=q, k=k, v=v, scales=scales, segments=_batch(case, lambda i: shared, case["past"]))
    if kind == "forward":
        layers, cos, sin = _forward_inputs(case, seed)
        shared = {i: x.past for i, x in enumerate(layers)} if case["past"] else None
        return dict(case=case, layers=layers, cos=cos, sin=sin, shared=shared)
    if kind == "fp8":
        x, w, b = _fp8_inputs(case, seed)
        lin = torch.nn.Linear(case["k"], case["n"], bias=case["bias"], device="cuda", dtype=w.dtype)
        with torch.no_grad():
            lin.weight.copy_(w)
            if case["bias"]:
                lin.bias.copy_(b)
        return dict(case=case, x=x, linear=FP8Linear(lin, case["rowwise"]))
    p, x, pasts = _deltanet_inputs(case, seed)
    cfg = SimpleNamespace(linear_num_key_heads=case["k_heads"], linear_num_value_heads=case["v_heads"],
                          linear_key_head_dim=128, linear_value_head_dim=case["v_dim"], linear_conv_kernel_dim=4,
                          hidden_size=case["hidden"], rms_norm_eps=1e-6)
    with torch.device("cuda"):
        layer = DeltaNet(cfg, 0).to(DTYPES[case["dtype"]])
    layer.load_state_dict(p)
    return dict(case=case, layer=layer, x=x, segments=_batch(case, lambda i: {0: pasts[i]} if pasts[i] else None, 64))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attend":
        segs = state["segments"]
        out = attend(state["q"], state["k"], state["v"], segs, 0, **state["scales"])
        return [out] + [t for s in segs if s.save for t in s.saved[0]]
    with torch.no_grad():
        if kind == "forward":
            segs = _batch(case, lambda i: state["shared"], case["past"])
            norm = None if case["norm"] == "none" else case["norm"]
            h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
            outs = []
            for i, x in enumerate(state["layers"]):
                q, k, v = x.qkv.view(-1, h + 2 * hkv, d).split((h, hkv, hkv), dim=1)
                q, k, v = qkv_front(q, k, v, state["cos"], state["sin"], q_norm_weight=x.qw, k_norm_weight=x.kw, norm=norm,
                                    segments=segs, layer=i)
                outs.append(attend(q, k, v, segs, i, save=False))
            return outs + [t for s in segs if s.save for i in range(case["layers"]) for t in s.saved[i]]
        if kind == "fp8":
            return state["linear"](state["x"])
        segs = state["segments"]
        out = state["layer"](state["x"], segs)
        return [out] + [t for s in segs if s.save for t in s.saved[0]]


# ------------------------------------------------------------------ what a pass cannot do without


def _attend_work(case):
    h, hkv, d, p = case["heads"], case["kv_heads"], case["head_dim"], case["past"]
    reqs = _structure(case)
    pairs = sum(t * p + t * (t + 1) // 2 + sum(b * (p + t) + b * (b + 1) // 2 for b in ls) for t, ls in reqs)
    es = {"fp32": 4, "e4m3": 1}.get(case["dtype"], 2)
    n, rows = _tokens(case), (max(1, reqs[-1][0] // 2) if case["save"] else 0)
    nbytes = (n * h + 2 * (n + p) * hkv) * d * es + n * h * d * max(es, 2) + 2 * rows * hkv * d * es
    return nbytes, 4 * d * h * pairs


def work(case):
    kind = case["kind"]
    if kind == "attend":
        nbytes, flops = _attend_work(case)
    elif kind == "forward":
        nbytes, flops = _attend_work(case)
        n, h, hkv, d = _tokens(case), case["heads"], case["kv_heads"], case["head_dim"]
        front = (2 * n * (h + hkv) * d + 2 * n * case["rotary"]) * 2  # q and k in and out, the tables
        nbytes, flops = case["layers"] * (nbytes + front), case["layers"] * flops
    elif kind == "fp8":
        m, n, k = case["tokens"], case["n"], case["k"]
        nbytes, flops = 2 * m * k + n * k + 2 * m * n + 4 * n, 2 * m * n * k
    else:
        n, hidden, hv, dv = _tokens(case), case["hidden"], case["v_heads"], case["v_dim"]
        conv, reqs = 2 * case["k_heads"] * 128 + hv * dv, len(_structure(case))
        weights = hidden * (conv + 2 * hv * dv + 2 * hv)
        states = (reqs if case["past"] else 0) + (1 if case["save"] else 0)
        nbytes = 4 * n * hidden + 2 * weights + 4 * states * hv * 128 * dv
        flops = 2 * n * weights + 2 * 4 * n * conv + 7 * n * hv * 128 * dv
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the largest difference from ``exact`` that was measured
    (bf16: attend and fp8 1.7e-3, forward 4.6e-3, deltanet 5.6e-3; fp32, whose
    q, k and P pass through fp16: 2.8e-4); fp16 has eight times bf16's
    precision, and accumulated rounding that the output type does not show."""
    rel = {"attend": 7e-3, "forward": 1.8e-2, "fp8": 7e-3, "deltanet": 2.2e-2}[case["kind"]]
    return {"rel": {"fp32": 1.2e-3, "fp16": rel / 4}.get(case["dtype"], rel)}


# ------------------------------------------------------------------ the same in 64 bits


def _attention64(case, q, k, v, past):
    """Tree attention of q [H, N, D] over k, v [Hkv, N, D] and the shared
    prefix's k, v [Hkv, P, D], all float64: causal within [past; trunk], and a
    branch sees past, trunk and itself."""
    h, n, d = q.shape
    rep = h // k.shape[0]
    out, start = torch.zeros_like(q), 0
    p = past[0].shape[1] if past else 0
    for trunk, lens in _structure(case):
        ids = torch.tensor(branch_ids(trunk, lens), device=q.device)
        end = start + len(ids)
        i = torch.arange(len(ids), device=q.device)
        own = (i[None] <= i[:, None]) & ((ids[None] == 0) | (ids[None] == ids[:, None]))
        hidden = torch.cat([own.new_zeros(len(ids), p), ~own], dim=1)
        for head in range(h):
            kh, vh = k[head // rep, start:end], v[head // rep, start:end]
            if past:
                kh, vh = torch.cat([past[0][head // rep], kh]), torch.cat([past[1][head // rep], vh])
            s = (q[head, start:end] @ kh.T.contiguous()) * d ** -0.5
            out[head, start:end] = torch.softmax(s.masked_fill_(hidden, -math.inf), dim=-1) @ vh
        start = end
    return out


def _saved64(case, k, v):
    """The saving request's first rows of k and v."""
    if not case["save"]:
        return []
    reqs = _structure(case)
    start = sum(t + sum(ls) for t, ls in reqs[:-1])
    rows = slice(start, start + max(1, reqs[-1][0] // 2))
    return [k[:, rows], v[:, rows]]


def _quantize64(x, dim):
    """e4m3 codes of x (per row of ``dim`` -1, or per tensor) times their scale, in float64."""
    x = x.float()
    amax = x.abs().amax(dim=dim, keepdim=True) if dim is not None else x.abs().amax().reshape(1, 1)
    scale = amax.clamp(min=1e-12) / torch.full_like(amax, 448.0)
    return (x / scale).to(torch.float8_e4m3fn).double() * scale.double()


def _front64(case, x, weight, cos, sin):
    """q or k rows [N, heads, D] after the norm and the rotary, in float64."""
    x = x.double()
    if case["norm"] != "none":
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
        x = x * (weight.double() + (1.0 if case["norm"] == "zero_centered" else 0.0))
    r = case["rotary"]
    a, rest = x[..., :r], x[..., r:]
    rot = torch.cat([-a[..., r // 2:], a[..., :r // 2]], dim=-1)
    return torch.cat([a * cos.double()[:, None] + rot * sin.double()[:, None], rest], dim=-1).transpose(0, 1)


def _recurrence64(q, k, v, g, beta, lens, states):
    """The gated delta rule over runs of consecutive rows, all runs a token at a time: q, k [N, Hv, 128], v [N, Hv, Dv]."""
    n, hv, dv = v.shape
    start = torch.tensor([sum(lens[:i]) for i in range(len(lens))], device=q.device)
    length = torch.tensor(lens, device=q.device)
    out, s = torch.zeros_like(v), states.clone()
    q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) * 128 ** -0.5
    k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    order = torch.argsort(length, descending=True)
    live = sorted(lens, reverse=True)
    for t in range(live[0]):
        runs = order[:sum(1 for x in live if x > t)]
        rows = start[runs] + t
        sr = s[runs] * g[rows].exp()[..., None, None]
        seen = (sr * k[rows][..., None]).sum(-2)
        sr = sr + k[rows][..., None] * (beta[rows][..., None] * (v[rows] - seen))[..., None, :]
        out[rows] = (sr * q[rows][..., None]).sum(-2)
        s[runs] = sr
    return out, s


def _deltanet64(case, p, x, pasts):
    hk, hv, dv, kernel = case["k_heads"], case["v_heads"], case["v_dim"], 4
    p, x = {name: t.double() for name, t in p.items()}, x.double()
    qkv, z = x @ p["in_proj_qkv.weight"].T, x @ p["in_proj_z.weight"].T
    beta = torch.sigmoid(x @ p["in_proj_b.weight"].T)
    g = -p["A_log"].exp() * torch.nn.functional.softplus(x @ p["in_proj_a.weight"].T + p["dt_bias"])
    w, n = p["conv1d.weight"][:, 0], x.shape[0]
    # the trunks first, then every branch behind its trunk: runs of (rows, the kernel - 1 rows before them)
    trunks, branches, owner, start, saved = [], [], [], 0, []
    reqs = _structure(case)
    for i, (trunk, lens) in enumerate(reqs):
        hist = pasts[i][0].double() if pasts[i] else x.new_zeros(kernel - 1, qkv.shape[1])
        rows = torch.arange(start, start + trunk, device=x.device)
        trunks.append((rows, hist))
        at = start + trunk
        for length in lens:
            branches.append((torch.arange(at, at + length, device=x.device), torch.cat([hist, qkv[rows]])[-(kernel - 1):]))
            owner.append(i)
            at += length
        if _saving(case, i, len(reqs)):
            saved = [torch.cat([hist, qkv[rows[:max(1, trunk // 2)]]])[-(kernel - 1):], i, max(1, trunk // 2)]
        start = at
    out = x.new_zeros(n, hv, dv)

    def phase(runs, states):
        rows = torch.cat([r for r, _ in runs])
        conv = []
        for r, hist in runs:
            src = torch.cat([hist, qkv[r]])
            conv.append(sum(src[j:j + len(r)] * w[:, j] for j in range(kernel)))
        conv = torch.nn.functional.silu(torch.cat(conv))
        q, k, v = conv.split((hk * 128, hk * 128, hv * dv), dim=1)
        q, k = (t.reshape(-1, hk, 128).repeat_interleave(hv // hk, dim=1) for t in (q, k))
        o, s = _recurrence64(q, k, v.reshape(-1, hv, dv), g[rows], beta[rows], [len(r) for r, _ in runs], states)
        out[rows] = o
        return s

    init = torch.stack([e[1].double() if e else x.new_zeros(hv, 128, dv) for e in pasts])
    finals = phase(trunks, init)
    if saved:
        tail, i, rows = saved
        saved = [tail, phase([(trunks[i][0][:rows], trunks[i][1])], init[i:i + 1])[0]]
    if branches:
        phase(branches, finals[torch.tensor(owner, device=x.device)])
    y = out * torch.rsqrt(out.square().mean(-1, keepdim=True) + 1e-6) * p["norm.weight"]
    y = y * torch.nn.functional.silu(z.reshape(n, hv, dv))
    return [y.reshape(n, -1) @ p["out_proj.weight"].T] + saved


def exact(case, seed):
    kind = case["kind"]
    if kind == "attend":
        q, k, v, past = _attend_inputs(case, seed)
        kept = (k, v)
        if case["dtype"] == "e4m3":
            q, k, v = (_quantize64(t, None) for t in (q, k, v))
            past = tuple(_quantize64(t, None) for t in past) if past else None
        q, k, v = q.double(), k.double(), v.double()
        past = tuple(t.double() for t in past) if past else None
        return [_attention64(case, q, k, v, past)] + [t.double() for t in _saved64(case, *kept)]
    if kind == "forward":
        layers, cos, sin = _forward_inputs(case, seed)
        h, hkv, d = case["heads"], case["kv_heads"], case["head_dim"]
        outs, saved = [], []
        for x in layers:
            q, k, v = x.qkv.view(-1, h + 2 * hkv, d).split((h, hkv, hkv), dim=1)
            q, k = _front64(case, q, x.qw, cos, sin), _front64(case, k, x.kw, cos, sin)
            v = v.double().transpose(0, 1)
            outs.append(_attention64(case, q, k, v, tuple(t.double() for t in x.past) if x.past else None))
            saved += _saved64(case, k, v)
        return outs + saved
    if kind == "fp8":
        x, w, b = _fp8_inputs(case, seed)
        dim = -1 if case["rowwise"] else None
        y = _quantize64(x, dim) @ _quantize64(w, dim).T.contiguous()
        return y + b.double() if case["bias"] else y
    return _deltanet64(case, *_deltanet_inputs(case, seed))
