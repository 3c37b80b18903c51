"""Timed workloads of the attention hot path, through the public entry points.

Each case is one layer call of an engine that serves the hybrid (GQA + Gated
DeltaNet) or the dense (GQA only) models: a decode token, a prompt, a turn
over a cached prefix, a DeltaNet layer's token or prompt. Sizes span what an
engine sends: one sequence and a batch, contexts from a few hundred rows to
32k, prompts from a few tokens to 8k, lengths that are no multiple of any tile.

``exact`` restates each case in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import torch

import aila_amd as A

BF = torch.bfloat16
EPS = 1e-6
THETA = 1e6

# (query heads, KV heads, head dim) of the attention layers
HEADS = ((16, 8, 128), (32, 8, 128), (40, 8, 128), (16, 4, 256))
# (key heads, value heads) of the DeltaNet layers, 128 x 128 states
DELTA_HEADS = ((16, 16), (16, 32), (16, 48), (8, 32))
D_STATE = 128
CONV_K = 4
PAGE = 64


def listed():
    return [
        # one chat sequence early in its context: norm + RoPE + append + attention
        # of one token, where launches and latency are all there is
        {"name": "decode_one_short", "kind": "decode", "B": 1, "Hq": 16, "Hkv": 8, "D": 128, "pos": 611, "gated": False, "ragged": False},
        # one sequence deep in a long context, gated attention (packed q|gate)
        {"name": "decode_one_long", "kind": "decode", "B": 1, "Hq": 16, "Hkv": 4, "D": 256, "pos": 32767, "gated": True, "ragged": False},
        # a served batch at long context, every sequence at its own position
        {"name": "decode_batch_long", "kind": "decode", "B": 8, "Hq": 16, "Hkv": 4, "D": 256, "pos": 32767, "gated": True, "ragged": True},
        # continuous batching over a page pool: append + decode, ragged lengths
        {"name": "decode_paged", "kind": "paged", "B": 32, "Hq": 40, "Hkv": 8, "D": 128, "pos": 4001},
        # a short prompt of a dense model, rows also written to the cache
        {"name": "prefill_short", "kind": "prefill", "S": 213, "Hq": 32, "Hkv": 8, "D": 128, "gated": False},
        # an ordinary prompt of a dense model
        {"name": "prefill_2k", "kind": "prefill", "S": 2048, "Hq": 32, "Hkv": 8, "D": 128, "gated": False},
        # a long prompt of a hybrid model with the gated epilogue
        {"name": "prefill_8k_gated", "kind": "prefill", "S": 8191, "Hq": 16, "Hkv": 4, "D": 256, "gated": True},
        # the next turn of a conversation: a short input over a cached prefix
        {"name": "prefill_turn", "kind": "turn", "S": 250, "start": 7900, "Hq": 16, "Hkv": 4, "D": 256},
        # DeltaNet layer, one token for a served batch
        {"name": "delta_step", "kind": "delta_step", "B": 8, "Hk": 16, "Hv": 32},
        # DeltaNet layer over a short turn
        {"name": "delta_prompt_short", "kind": "delta_prompt", "B": 1, "T": 130, "Hk": 16, "Hv": 32},
        # DeltaNet layer over a long prompt
        {"name": "delta_prompt_4k", "kind": "delta_prompt", "B": 1, "T": 4096, "Hk": 16, "Hv": 32},
        # two prompts at once, three value heads to a key head
        {"name": "delta_prompt_48", "kind": "delta_prompt", "B": 2, "T": 1500, "Hk": 16, "Hv": 48},
    ]


# What one drawn case may cost at most: the largest listed one of its kind.
def _cost(case):
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    limits = {}
    for c in listed():
        limits[c["kind"]] = max(limits.get(c["kind"], 0.0), _cost(c))
    kind = rng.choice(sorted(limits))
    Hq, Hkv, D = rng.choice(HEADS)
    while True:
        if kind == "decode":
            case = {"kind": kind, "B": _log_int(rng, 1, 32), "Hq": Hq, "Hkv": Hkv, "D": D,
                    "pos": _log_int(rng, 16, 32767), "gated": D == 256, "ragged": rng.random() < 0.5}
        elif kind == "paged":
            case = {"kind": kind, "B": _log_int(rng, 1, 64), "Hq": Hq, "Hkv": Hkv, "D": D, "pos": _log_int(rng, 16, 16000)}
        elif kind == "prefill":
            case = {"kind": kind, "S": _log_int(rng, 8, 8191), "Hq": Hq, "Hkv": Hkv, "D": D, "gated": D == 256}
        elif kind == "turn":
            case = {"kind": kind, "S": _log_int(rng, 8, 600), "start": _log_int(rng, 200, 16000), "Hq": Hq, "Hkv": Hkv, "D": D}
        elif kind == "delta_step":
            Hk, Hv = rng.choice(DELTA_HEADS)
            case = {"kind": kind, "B": _log_int(rng, 1, 32), "Hk": Hk, "Hv": Hv}
        else:
            Hk, Hv = rng.choice(DELTA_HEADS)
            case = {"kind": kind, "B": rng.choice((1, 1, 2, 3)), "T": _log_int(rng, 8, 4096), "Hk": Hk, "Hv": Hv}
        if _cost(case) <= limits[kind]:
            return case


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rn(g, shape, std=1.0, dtype=BF):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _rn_big(g, shape):
    t = torch.empty(shape, device="cuda", dtype=BF)
    t.normal_(generator=g)
    return t


def _positions(case, seed):
    """Row of each sequence's new token: ragged batches have their own, the first at the bound."""
    B, pos = case["B"], case["pos"]
    g = torch.Generator()
    g.manual_seed(int(seed) + 77)
    p = (pos * (0.5 + 0.5 * torch.rand(B, generator=g))).to(torch.int32)
    p[0] = pos
    return p


def _capacity(rows):
    return -(-rows // 1024) * 1024


def prepare(case, seed):
    kind, g, s = case["kind"], _gen(seed), {"case": dict(case)}
    if kind == "decode":
        B, Hq, Hkv, D, pos = (case[k] for k in ("B", "Hq", "Hkv", "D", "pos"))
        cap = _capacity(pos + 1)
        s["k_cache"], s["v_cache"] = _rn_big(g, (B, Hkv, cap, D)), _rn_big(g, (B, Hkv, cap, D))
        s["q_in"] = _rn(g, (B, Hq, 2 * D if case["gated"] else D))
        s["k_new"], s["v_new"] = _rn(g, (B, Hkv, D)), _rn(g, (B, Hkv, D))
        s["qw"] = (1.2 + 0.2 * torch.randn(D, generator=g, device="cuda")).to(BF)
        s["kw"] = (1.0 + 0.2 * torch.randn(D, generator=g, device="cuda")).to(BF)
        s["positions"] = _positions(case, seed).cuda() if case["ragged"] else None
        s["out"] = torch.empty((B, Hq, D), device="cuda", dtype=BF)
        s["ws"] = torch.empty(A.gqa_decode_workspace_size(B, Hq, D), device="cuda", dtype=torch.uint8)
    elif kind == "paged":
        B, Hq, Hkv, D, pos = (case[k] for k in ("B", "Hq", "Hkv", "D", "pos"))
        rows = _positions(case, seed)
        mp = pos // PAGE + 1
        gc = torch.Generator()
        gc.manual_seed(int(seed) + 5)
        table = torch.randperm(B * mp, generator=gc).to(torch.int32).view(B, mp)
        s["k_pages"], s["v_pages"] = _rn_big(g, (B * mp, Hkv, PAGE, D)), _rn_big(g, (B * mp, Hkv, PAGE, D))
        s["q"] = _rn(g, (B, Hq, D), 1.2)
        s["k_new"], s["v_new"] = _rn(g, (B, Hkv, D)), _rn(g, (B, Hkv, D))
        s["table"], s["rows"] = table.cuda(), rows.cuda()
        s["lens"] = s["rows"] + 1
        s["out"] = torch.empty((B, Hq, D), device="cuda", dtype=BF)
        s["ws"] = torch.empty(A.gqa_decode_workspace_size(B, Hq, D), device="cuda", dtype=torch.uint8)
    elif kind == "prefill":
        S, Hq, Hkv, D = (case[k] for k in ("S", "Hq", "Hkv", "D"))
        cap = _capacity(S)
        s["q"], s["k"], s["v"] = _rn(g, (S, Hq * D), 1.2), _rn(g, (S, Hkv * D)), _rn(g, (S, Hkv * D))
        s["gate"] = _rn(g, (S, Hq * D)) if case["gated"] else None
        s["k_cache"] = torch.zeros((Hkv, cap, D), device="cuda", dtype=BF)
        s["v_cache"] = torch.zeros((Hkv, cap, D), device="cuda", dtype=BF)
        s["out"] = torch.empty((S, Hq * D), device="cuda", dtype=BF)
        s["gated"] = torch.empty((S, Hq * D), device="cuda", dtype=BF) if case["gated"] else None
    elif kind == "turn":
        S, start, Hq, Hkv, D = (case[k] for k in ("S", "start", "Hq", "Hkv", "D"))
        cap = _capacity(start + S)
        s["q"], s["k"], s["v"] = _rn(g, (S, Hq * D), 1.2), _rn(g, (S, Hkv * D)), _rn(g, (S, Hkv * D))
        s["k_cache"], s["v_cache"] = _rn_big(g, (Hkv, cap, D)), _rn_big(g, (Hkv, cap, D))
        s["out"] = torch.empty((S, Hq * D), device="cuda", dtype=BF)
        n = A.gqa_prefill_cached_workspace_size(S, start, Hq, Hkv, D)
        s["ws"] = torch.empty(n, device="cuda", dtype=torch.uint8) if n else None
    else:
        B, Hk, Hv, d = case["B"], case["Hk"], case["Hv"], D_STATE
        T = case.get("T", 1)
        ch, zd = 2 * Hk * d + Hv * d, Hv * d
        # the projection's fused rows [qkv | z | a | b], padded to 16 bytes
        width = -(-(ch + zd + 2 * Hv) // 8) * 8
        rows = _rn(g, (B, T, width))
        if kind == "delta_step":
            rows = rows[:, 0]
        s["qkv"], s["z"] = rows[..., :ch], rows[..., ch:ch + zd]
        s["a"], s["b"] = rows[..., ch + zd:ch + zd + Hv], rows[..., ch + zd + Hv:ch + zd + 2 * Hv]
        s["conv_w"] = _rn(g, (ch, CONV_K), 0.5)
        s["conv_state"] = torch.randn((B, CONV_K - 1, ch), generator=g, device="cuda").to(BF).float()
        s["norm_w"] = 1.0 + 0.1 * torch.randn(d, generator=g, device="cuda")
        # gates as such layers are initialised: A in [1, 16], steps of 0.001 to 0.1
        s["A_log"] = (1.0 + 15.0 * torch.rand(Hv, generator=g, device="cuda")).log()
        dt = torch.exp(math.log(1e-3) + math.log(100.0) * torch.rand(Hv, generator=g, device="cuda"))
        s["dt_bias"] = (dt + torch.log(-torch.expm1(-dt))).to(BF)
        s["state"] = torch.randn((B, Hv, d, d), generator=g, device="cuda") * 0.1
        if kind == "delta_step":
            s["arrivals"] = torch.zeros(B * Hk, device="cuda", dtype=torch.int32)
            s["out"] = torch.empty((B, zd), device="cuda", dtype=BF)
        else:
            s["ws"] = torch.empty(A.deltanet_layer_prefill_workspace_size(B, T, Hk, Hv), device="cuda", dtype=torch.uint8)
            s["out"] = torch.empty((B, T, zd), device="cuda", dtype=BF)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "decode":
        out = A.gqa_decode_prepare_append(
            s["q_in"], s["k_new"], s["v_new"], s["k_cache"], s["v_cache"], c["pos"], q_norm_w=s["qw"], k_norm_w=s["kw"],
            rotary_dim=c["D"] // 4 if c["gated"] else c["D"], theta=THETA, eps=EPS, packed_gate=c["gated"],
            out=s["out"], workspace=s["ws"], positions=s["positions"], apply_gate=c["gated"])
        return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "paged":
        A.kv_append_paged(s["k_new"], s["v_new"], s["k_pages"], s["v_pages"], s["table"], s["rows"])
        out = A.gqa_decode_paged(s["q"], s["k_pages"], s["v_pages"], s["table"], s["lens"], c["pos"] + 1, out=s["out"], workspace=s["ws"])
        return {"out": out, "k_pages": s["k_pages"], "v_pages": s["v_pages"]}
    if kind == "prefill":
        out = A.gqa_prefill(s["q"], s["k"], s["v"], c["Hq"], c["Hkv"], out=s["out"], k_cache=s["k_cache"], v_cache=s["v_cache"])
        r = {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
        if c["gated"]:
            r["gated"] = A.sigmoid_mul(out, s["gate"], out=s["gated"])
        return r
    if kind == "turn":
        A.copy_to_cache(s["k"], s["k_cache"], c["start"])
        A.copy_to_cache(s["v"], s["v_cache"], c["start"])
        out = A.gqa_prefill_cached(s["q"], s["k_cache"], s["v_cache"], c["start"], c["Hq"], out=s["out"], workspace=s["ws"])
        return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "delta_step":
        out = A.deltanet_layer_decode(s["qkv"], s["z"], s["a"], s["b"], s["conv_w"], s["conv_state"], 0, s["norm_w"], s["state"],
                                      c["Hk"], out=s["out"], dt_bias=s["dt_bias"], A_log=s["A_log"], eps=EPS, arrivals=s["arrivals"])
    else:
        out = A.deltanet_layer_prefill(s["qkv"], s["z"], s["a"], s["b"], s["conv_w"], s["conv_state"], 0, s["norm_w"], s["state"],
                                       c["Hk"], out=s["out"], workspace=s["ws"], dt_bias=s["dt_bias"], A_log=s["A_log"], eps=EPS)
    return {"out": out, "state": s["state"], "conv_state": s["conv_state"]}


def _mean_rows(case):
    """Rows attended by the whole batch (ragged: its expected sum)."""
    B, n = case["B"], case["pos"] + 1
    if case["kind"] == "paged" or case["ragged"]:
        return n + 0.75 * n * (B - 1)
    return B * n


def work(case):
    kind = case["kind"]
    if kind in ("decode", "paged"):
        B, Hq, Hkv, D = (case[k] for k in ("B", "Hq", "Hkv", "D"))
        rows = _mean_rows(case)
        q = Hq * D * (2 if case.get("gated") else 1)
        return {"bytes": rows * Hkv * D * 4 + B * (q + Hq * D) * 2 + B * Hkv * D * 8, "flops": 4 * rows * Hq * D}
    if kind == "prefill":
        S, Hq, Hkv, D = (case[k] for k in ("S", "Hq", "Hkv", "D"))
        return {"bytes": 2 * S * D * ((5 if case["gated"] else 2) * Hq + 4 * Hkv), "flops": 2 * D * Hq * S * (S + 1)}
    if kind == "turn":
        S, start, Hq, Hkv, D = (case[k] for k in ("S", "start", "Hq", "Hkv", "D"))
        return {"bytes": 4 * S * Hq * D + 4 * (start + 3 * S) * Hkv * D, "flops": 4 * D * Hq * (S * start + S * (S + 1) / 2)}
    B, Hk, Hv, d = case["B"], case["Hk"], case["Hv"], D_STATE
    T = case.get("T", 1)
    ch = 2 * Hk * d + Hv * d
    # state, fused rows, output, conv ring and weights; the recurrence's three
    # products with the state per token (S^T k, k d^T, S^T q) and the conv
    return {"bytes": B * Hv * d * d * 8 + B * T * (2 * ch + 4 * Hv * d + 4 * Hv) + B * 6 * 4 * ch + ch * CONV_K * 2,
            "flops": B * T * (6 * Hv * d * d + 2 * CONV_K * ch)}


def tolerance(case):
    # four times the largest error against 64 bits that a sweep of the ranges
    # shows: outputs are rounded to bf16 (2-norm error about 1.7e-3; the
    # rounded probabilities of a prompt's attention bring it to about 3e-3),
    # recurrent states are fp32
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------- 64 bits ----
def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, pos, rot):
    """NeoX rotation of x [..., D] at positions pos (broadcast against x[..., 0])."""
    half = rot // 2
    ang = pos[..., None].double() * THETA ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / rot)
    c, n = ang.cos(), ang.sin()
    a, b = x[..., :half], x[..., half:rot]
    return torch.cat((a * c - b * n, b * c + a * n, x[..., rot:]), -1)


def _attend(q, k, v, first):
    """q [S, Hq, D] at rows first.. over k, v [Hkv, L, D], causal, fp64."""
    S, Hq, D = q.shape
    Hkv, L, _ = k.shape
    G = Hq // Hkv
    out = torch.empty_like(q)
    cols = torch.arange(L, device=q.device)
    for h in range(Hq):
        kt = k[h // G].t().contiguous()
        for i in range(0, S, 2048):
            sc = (q[i:i + 2048, h].contiguous() @ kt) / math.sqrt(D)
            row = first + i + torch.arange(sc.shape[0], device=q.device)
            sc.masked_fill_(cols[None] > row[:, None], -math.inf)
            out[i:i + 2048, h] = torch.softmax(sc, -1) @ v[h // G]
    return out


def _delta(s, c):
    B, Hk, Hv, d = c["B"], c["Hk"], c["Hv"], D_STATE
    T, R = c.get("T", 1), CONV_K - 1
    ch = 2 * Hk * d + Hv * d
    x = s["qkv"].double().reshape(B, T, ch)
    hist = torch.cat((s["conv_state"].double(), x), 1)              # ring head 0: row 0 is the oldest
    w = s["conv_w"].double()
    y = sum(hist[:, j:j + T] * w[:, j] for j in range(CONV_K))
    y = y * torch.sigmoid(y)
    q, k, v = y.split((Hk * d, Hk * d, Hv * d), -1)
    norm = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + EPS)  # noqa: E731
    q = norm(q.reshape(B, T, Hk, d)).repeat_interleave(Hv // Hk, 2)
    k = norm(k.reshape(B, T, Hk, d)).repeat_interleave(Hv // Hk, 2)
    v = v.reshape(B, T, Hv, d)
    beta = torch.sigmoid(s["b"].double().reshape(B, T, Hv))
    decay = torch.exp(-torch.nn.functional.softplus(s["a"].double().reshape(B, T, Hv) + s["dt_bias"].double()) * s["A_log"].double().exp())
    S = s["state"].double()
    o = torch.empty((B, T, Hv, d), device=x.device, dtype=torch.float64)
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        kt = k[:, t]
        u = (v[:, t] - (S * kt[..., None]).sum(-2)) * beta[:, t, :, None]
        S = S + kt[..., None] * u[..., None, :]
        o[:, t] = (S * q[:, t][..., None]).sum(-2)
    o = o / math.sqrt(d)
    z = s["z"].double().reshape(B, T, Hv, d)
    o = _rms(o, s["norm_w"].double()) * z * torch.sigmoid(z)
    ring = s["conv_state"].double().clone()
    for t in range(max(0, T - R), T):
        ring[:, t % R] = x[:, t]
    shape = (B, Hv * d) if c["kind"] == "delta_step" else (B, T, Hv * d)
    return {"out": o.reshape(shape), "state": S, "conv_state": ring}


def exact(case, seed):
    s, c = prepare(case, seed), case
    kind = c["kind"]
    if kind == "decode":
        B, Hq, Hkv, D, pos = (c[k] for k in ("B", "Hq", "Hkv", "D", "pos"))
        rot = D // 4 if c["gated"] else D
        rows = s["positions"].tolist() if c["ragged"] else [pos] * B
        p = torch.tensor(rows, device="cuda")[:, None]
        q = _rope(_rms(s["q_in"][..., :D].double(), s["qw"].double()), p, rot)
        kn = _rope(_rms(s["k_new"].double(), s["kw"].double()), p, rot)
        out = torch.empty((B, Hq, D), device="cuda", dtype=torch.float64)
        k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
        for b, r in enumerate(rows):
            k_cache[b, :, r], v_cache[b, :, r] = kn[b], s["v_new"][b].double()
            out[b] = _attend(q[b][None], k_cache[b, :, :r + 1], v_cache[b, :, :r + 1], r)[0]
        if c["gated"]:
            out = out * torch.sigmoid(s["q_in"][..., D:].double())
        return {"out": out, "k_cache": k_cache, "v_cache": v_cache}
    if kind == "paged":
        B, Hq, D = c["B"], c["Hq"], c["D"]
        out = torch.empty((B, Hq, D), device="cuda", dtype=torch.float64)
        k_pages, v_pages = s["k_pages"].double(), s["v_pages"].double()
        for b, r in enumerate(s["rows"].tolist()):
            t = s["table"][b].long()
            k_pages[t[r // PAGE], :, r % PAGE], v_pages[t[r // PAGE], :, r % PAGE] = s["k_new"][b].double(), s["v_new"][b].double()
            n = r // PAGE + 1
            k, v = (x[t[:n]].transpose(0, 1).reshape(c["Hkv"], n * PAGE, D)[:, :r + 1] for x in (k_pages, v_pages))
            out[b] = _attend(s["q"][b].double()[None], k, v, r)[0]
        return {"out": out, "k_pages": k_pages, "v_pages": v_pages}
    if kind in ("prefill", "turn"):
        S, Hq, Hkv, D = (c[k] for k in ("S", "Hq", "Hkv", "D"))
        start = c.get("start", 0)
        k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
        k_cache[:, start:start + S] = s["k"].double().view(S, Hkv, D).transpose(0, 1)
        v_cache[:, start:start + S] = s["v"].double().view(S, Hkv, D).transpose(0, 1)
        out = _attend(s["q"].double().view(S, Hq, D), k_cache[:, :start + S], v_cache[:, :start + S], start).reshape(S, Hq * D)
        r = {"out": out, "k_cache": k_cache, "v_cache": v_cache}
        if kind == "prefill" and c["gated"]:
            r["gated"] = out * torch.sigmoid(s["gate"].double())
        return r
    return _delta(s, c)
