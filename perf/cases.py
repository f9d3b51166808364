"""The work a user has this framework do, as cases that can be timed and checked.

A case is one call of a public entry point: the layer forward
(``GatedSparseAttention``), or one of the launchers and sub-modules that the
reference's own code calls (``fused_sparse_attention``, ``fused_gated_indexer``,
``AdaptiveTopKSelector``, ``apply_rotary_pos_emb``).  All are forward only: the
framework has no backward.  Sizes are the layer's own (D=2048, H=16, d=128, an
indexer of 4 heads of 64), the sequence lengths those of the benchmark's configs
and the harness's sweep, and ragged ones between them.
"""

import math

import torch

from gsa_gdn_benchmarkstudy_amd import gsa

D, H, DH, HI, DI = 2048, 16, 128, 4, 64
K_MIN, K_MAX = 256, 4096


def _layer(name, dtype, B, T, k_base=2048, k_min=K_MIN, k_max=K_MAX, mode="fixed"):
    return {"name": name, "op": "layer", "dtype": dtype, "B": B, "T": T, "k_base": k_base, "k_min": k_min,
            "k_max": k_max, "mode": mode}


def listed():
    return [
        # the harness sweep's shortest sequence: launches and host time count
        _layer("layer_bf16_T512", "bf16", 1, 512),
        # a short prompt (benchmark config c2)
        _layer("layer_bf16_T4096", "bf16", 1, 4096),
        # a ragged batch: nothing is a multiple of a tile
        _layer("layer_bf16_B2_T3001", "bf16", 2, 3001),
        # the benchmark's headline (c3)
        _layer("layer_bf16_T16384", "bf16", 1, 16384),
        # a batch whose sequences differ in scale, with the variance-based k (c4)
        _layer("layer_bf16_B4_T8192_var", "bf16", 4, 8192, mode="variance"),
        # long context (c5), the largest
        _layer("layer_bf16_T65536", "bf16", 1, 65536),
        # full precision, with the selector of the fp32 config (c1) on a longer sequence
        _layer("layer_f32_T2048", "f32", 1, 2048, k_base=256, k_min=64, k_max=512),
        # the attention launcher on its own, fed as the reference's forward feeds it
        # (the selected keys sorted ascending)
        {"name": "attn_bf16_T8192", "op": "attn", "dtype": "bf16", "B": 1, "T": 8192, "k": 2048, "ascending": True},
        # the same in fp32, ragged, fed with the selector's own order (by score)
        {"name": "attn_f32_B2_T1537", "op": "attn", "dtype": "f32", "B": 2, "T": 1537, "k": 256, "ascending": False},
        # the indexer's full score matrix (the reference's launcher)
        {"name": "scores_bf16_T8192", "op": "scores", "dtype": "bf16", "B": 1, "T": 8192, "causal": True},
        # the selector on such a matrix
        {"name": "topk_T8192_k2048", "op": "topk", "B": 1, "T": 8192, "k_base": 2048},
        # RoPE of q and k
        {"name": "rope_bf16_B2_T8192", "op": "rope", "dtype": "bf16", "B": 2, "T": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["layer", "layer", "layer", "layer_f32", "attn", "attn", "scores", "topk", "rope"])
    if op == "layer":
        B = rng.choice([1, 1, 1, 2, 3, 4])
        c = _layer("", "bf16", B, _log_int(rng, 200, 32768 // B), mode=rng.choice(["fixed", "fixed", "variance"]))
    elif op == "layer_f32":
        c = _layer("", "f32", rng.choice([1, 1, 2]), _log_int(rng, 200, 3000), k_base=256, k_min=64, k_max=512)
    elif op == "attn":
        f32 = rng.random() < 0.4
        T = _log_int(rng, 200, 3000 if f32 else 8192)
        c = {"op": "attn", "dtype": "f32" if f32 else "bf16", "B": rng.choice([1, 1, 2]), "T": T,
             "k": min(T, _log_int(rng, 128, 512 if f32 else 2048)), "ascending": rng.random() < 0.5}
    elif op == "scores":
        c = {"op": "scores", "dtype": rng.choice(["bf16", "bf16", "f32"]), "B": rng.choice([1, 2]),
             "T": _log_int(rng, 200, 8192), "causal": rng.random() < 0.8}
    elif op == "topk":
        c = {"op": "topk", "B": rng.choice([1, 2]), "T": _log_int(rng, 200, 8192),
             "k_base": rng.choice([256, 1024, 2048])}
    else:
        c = {"op": "rope", "dtype": rng.choice(["bf16", "bf16", "f32"]), "B": rng.choice([1, 2, 4]),
             "T": _log_int(rng, 200, 8192)}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _layer_inputs(case, seed):
    """The layer's weights by name and its input: weights N(0, 0.02), gate biases 0.5,
    other biases 0, x ~ N(0, 1), in a batch scaled per sequence by U(0.5, 2)."""
    dt, g = _DTYPES[case["dtype"]], _gen(seed)
    w = {}
    for name, rows in (("q_proj", D), ("k_proj", D), ("v_proj", D), ("o_proj", D),
                       ("value_gate.gate_proj", D), ("output_gate.gate_proj", D),
                       ("indexer.idx_q_proj", HI * DI), ("indexer.idx_k_proj", DI), ("indexer.idx_w_proj", HI)):
        w[name + ".weight"] = (_randn(g, rows, D) * 0.02).to(dt)
    for name in ("value_gate", "output_gate"):
        w[name + ".gate_proj.bias"] = torch.full((D,), 0.5, device="cuda", dtype=dt)
    w["indexer.idx_w_proj.bias"] = torch.zeros(HI, device="cuda", dtype=dt)
    w["indexer.idx_bias"] = torch.zeros(HI, device="cuda", dtype=dt)
    x = _randn(g, case["B"], case["T"], D)
    if case["B"] > 1:
        x *= 0.5 + 1.5 * torch.rand(case["B"], 1, 1, generator=g, device="cuda")
    return w, x.to(dt)


def _indexer_inputs(case, seed):
    """q_idx, k_idx, w as the indexer's projections of a unit-variance input give them."""
    dt, g = _DTYPES[case.get("dtype", "bf16")], _gen(seed)
    B, T = case["B"], case["T"]
    s = 0.02 * math.sqrt(D)
    return ((_randn(g, B, T, HI, DI) * s).to(dt), (_randn(g, B, T, DI) * s).to(dt), (_randn(g, B, T, HI) * s).to(dt))


def _scores(q, k, w, causal, dtype):
    """The indexer's scores in plain torch: sum_h sigmoid(w_h) sigmoid(q_h . k / 8)."""
    B, T = q.shape[:2]
    q, k, w = q.to(dtype), k.to(dtype), w.to(dtype)
    s = torch.zeros(B, T, T, device="cuda", dtype=dtype)
    for b in range(B):
        for h in range(HI):
            z = (q[b, :, h] @ k[b].t().contiguous()).mul_(DI ** -0.5)
            s[b] += z.sigmoid_().mul_(torch.sigmoid(w[b, :, h, None]))
    if causal:
        s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device="cuda").triu_(1), -math.inf)
    return s


def _attn_inputs(case, seed):
    """q, k, v ~ N(0, 1) and a causal selection: min(t + 1, k) random keys of row t; the
    entries past them name later keys and are masked out, as the selector leaves them."""
    dt, g = _DTYPES[case["dtype"]], _gen(seed)
    B, T, K = case["B"], case["T"], case["k"]
    q, k, v = (_randn(g, B, T, H, DH, dtype=dt) for _ in range(3))
    later = torch.ones(T, T, dtype=torch.bool, device="cuda").triu_(1)
    r = torch.rand(B, T, T, generator=g, device="cuda").masked_fill_(later, -1.0)
    idx = r.topk(K, dim=-1).indices
    del r, later
    if case["ascending"]:
        idx = idx.sort(dim=-1).values
    mask = idx <= torch.arange(T, device="cuda")[None, :, None]
    return q, k, v, idx, mask


def _rope_inputs(case, seed):
    dt, g = _DTYPES[case["dtype"]], _gen(seed)
    B, T = case["B"], case["T"]
    q, k = (_randn(g, B, T, H, DH, dtype=dt) for _ in range(2))
    cos, sin = _rope_tables(T, dt)
    return q, k, cos[None, :, None], sin[None, :, None]


def _rope_tables(T, dt):
    """cos and sin of t * 10000^(-2i/128), the fp32 angles repeated over both halves."""
    inv = 1.0 / (10000.0 ** (torch.arange(0, DH, 2).float() / DH))
    ang = torch.outer(torch.arange(T).float(), inv)
    ang = torch.cat((ang, ang), dim=-1)
    return ang.cos().to("cuda").to(dt), ang.sin().to("cuda").to(dt)


# ---------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------

def prepare(case, seed):
    op = case["op"]
    if op == "layer":
        w, x = _layer_inputs(case, seed)
        m = gsa.GatedSparseAttention(D, H, k_max=min(case["k_max"], case["T"]), d_indexer=DI, n_idx_heads=HI,
                                     k_base=case["k_base"], k_min=case["k_min"])
        m = m.to("cuda").to(_DTYPES[case["dtype"]]).eval()
        m.load_state_dict(w, strict=False)      # the RoPE frequencies stay the module's own
        m.topk_selector.mode = case["mode"]
        m.fuse_projections()
        return {"op": op, "layer": m, "x": x}
    if op == "attn":
        return {"op": op, "args": (*_attn_inputs(case, seed), DH ** -0.5)}
    if op == "scores":
        bias = torch.zeros(HI, device="cuda", dtype=_DTYPES[case["dtype"]])
        return {"op": op, "args": (*_indexer_inputs(case, seed), bias, DI ** -0.5, case["causal"])}
    if op == "topk":
        return {"op": op, "select": gsa.AdaptiveTopKSelector(k_base=case["k_base"], k_min=K_MIN, k_max=K_MAX),
                "scores": _scores(*_indexer_inputs(case, seed), True, torch.float32)}
    return {"op": op, "args": _rope_inputs(case, seed)}


def run(state):
    op = state["op"]
    with torch.no_grad():
        if op == "layer":
            return state["layer"](state["x"])
        if op == "attn":
            return gsa.fused_sparse_attention(*state["args"])
        if op == "scores":
            return gsa.fused_gated_indexer(*state["args"])
        if op == "topk":
            return state["select"](state["scores"])
        return gsa.apply_rotary_pos_emb(*state["args"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _pairs(B, T, k):
    """Selected (row, key) pairs: B * sum_t min(t + 1, k)."""
    k = min(k, T)
    return B * (k * (k + 1) // 2 + (T - k) * k)


def work(case):
    op, B, T = case["op"], case["B"], case["T"]
    s = 2 if case.get("dtype") == "bf16" else 4
    pairs = B * T * (T + 1) // 2 if case.get("causal", True) else B * T * T
    if op == "layer":
        # projections, causal indexer products, attention over the selected pairs, o_proj
        n_proj = 5 * D + HI * DI + DI + HI
        flops = 2 * B * T * D * (n_proj + D) + 2 * HI * DI * pairs + 4 * H * DH * _pairs(B, T, case["k_base"])
        return {"bytes": s * (2 * B * T * D + D * (n_proj + D)), "flops": flops}
    if op == "attn":
        p = _pairs(B, T, case["k"])
        return {"bytes": s * 4 * B * T * H * DH + 9 * B * T * case["k"], "flops": 4 * H * DH * p}
    if op == "scores":
        return {"bytes": s * B * T * (HI * DI + DI + HI) + 4 * B * T * T, "flops": 2 * HI * DI * pairs}
    if op == "topk":
        return {"bytes": 4 * B * T * T + 9 * B * T * min(case["k_base"], T), "flops": 0}
    return {"bytes": s * (4 * B * T * H * DH + 2 * T * DH), "flops": 6 * B * T * H * DH}


# About four times the relative error measured against ``exact`` (layer: bf16
# 0.0046-0.0076, fp32 0.0016; attention: bf16 0.0015, fp32 3.2e-7; scores
# 7.1e-8; RoPE in bf16 0.0024).  The layer's is wider than its arithmetic: an
# ulp of a projection moves keys at the edge of a row's selection.  The
# selector's indices, mask and width are whole numbers with one right answer.
def tolerance(case):
    op, bf16 = case["op"], case.get("dtype") == "bf16"
    if op == "topk":
        return "exact"
    if op == "layer":
        return {"rel": 2e-2} if bf16 else {"rel": 6e-3}
    if op == "attn":
        return {"rel": 6e-3} if bf16 else {"rel": 2e-6}
    if op == "scores":
        return {"rel": 1e-6}
    return {"rel": 1e-2} if bf16 else {"rel": 1e-6}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _rope64(x, cos, sin):
    half = DH // 2
    return x * cos[:, None, :] + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin[:, None, :]


def _attend64(q, k, v, sel, r0):
    """softmax(q k^T / sqrt(d)) v over the keys that sel [rows, T] holds, one head at a time."""
    out = torch.empty_like(q)
    for h in range(H):
        z = (q[:, h] @ k[:, h].t().contiguous()).mul_(DH ** -0.5).masked_fill_(~sel, -math.inf)
        out[:, h] = torch.softmax(z, dim=-1) @ v[:, h].contiguous()
    return out


def _layer64(case, seed):
    """The layer with 64-bit arithmetic.  The projections are stored in the case's type, as
    the layer defines them (in bf16 their rounding decides which keys a row selects)."""
    w, x = _layer_inputs(case, seed)
    dt = _DTYPES[case["dtype"]]
    w64 = {n: t.double() for n, t in w.items()}
    B, T = case["B"], case["T"]
    cos, sin = _layer_tables(case)
    out = torch.empty(B, T, D, device="cuda", dtype=torch.float64)

    def store(t):
        return t.to(dt).double() if case["dtype"] == "bf16" else t

    for b in range(B):
        xb = x[b].double()

        def proj(name):
            y = xb @ w64[name + ".weight"].t().contiguous()
            if name + ".bias" in w64:
                y += w64[name + ".bias"]
            return store(y)

        q, k, v = (proj(n).view(T, H, DH) for n in ("q_proj", "k_proj", "v_proj"))
        v = v * torch.sigmoid(proj("value_gate.gate_proj")).view(T, H, DH)
        og = torch.sigmoid(proj("output_gate.gate_proj")).view(T, H, DH)
        q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
        iq, ik = proj("indexer.idx_q_proj").view(T, HI, DI), proj("indexer.idx_k_proj")
        iw = torch.sigmoid(proj("indexer.idx_w_proj"))
        n_k = min(case["k_base"], case["k_max"], T)
        att = torch.empty(T, H, DH, device="cuda", dtype=torch.float64)
        for r0 in range(0, T, 2048):
            r1 = min(T, r0 + 2048)
            s = torch.zeros(r1 - r0, T, device="cuda", dtype=torch.float64)
            for h in range(HI):
                z = (iq[r0:r1, h] @ ik.t().contiguous()).mul_(DI ** -0.5)
                s += z.sigmoid_().mul_(iw[r0:r1, h, None])
            later = torch.arange(T, device="cuda")[None, :] > torch.arange(r0, r1, device="cuda")[:, None]
            s.masked_fill_(later, -math.inf)
            sel = (s >= s.topk(n_k, dim=-1).values[:, -1:]) & ~later
            att[r0:r1] = _attend64(q[r0:r1], k, v, sel, r0)
        out[b] = (att * og).reshape(T, D) @ w64["o_proj.weight"].t().contiguous()
    return out


def _layer_tables(case):
    """The RoPE tables as the layer stores them: 8192 rows from fp32 frequencies, cast; a
    longer sequence's from the frequencies in the layer's type."""
    T, dt = case["T"], _DTYPES[case["dtype"]]
    inv = 1.0 / (10000.0 ** (torch.arange(0, DH, 2).float() / DH))
    if T > 8192:
        inv = inv.to(dt)
    ang = torch.outer(torch.arange(T, dtype=torch.float32), inv)
    ang = torch.cat((ang, ang), dim=-1)
    return tuple(t.to("cuda").to(dt).double() for t in (ang.cos(), ang.sin()))


def exact(case, seed):
    op = case["op"]
    if op == "layer":
        # the variance-based k depends on floors of a global mean; past 16384 keys it takes too long
        if case["mode"] != "fixed" or case["T"] > 16384:
            return None
        return _layer64(case, seed)
    if op == "attn":
        q, k, v, idx, mask = _attn_inputs(case, seed)
        out = torch.empty(*q.shape, device="cuda", dtype=torch.float64)
        for b in range(case["B"]):
            for r0 in range(0, case["T"], 2048):
                r = slice(r0, min(case["T"], r0 + 2048))
                sel = torch.zeros(r.stop - r0, case["T"], dtype=torch.bool, device="cuda")
                sel.scatter_(1, idx[b, r], mask[b, r])
                out[b, r] = _attend64(q[b, r].double(), k[b].double(), v[b].double(), sel, r0)
        return out
    if op == "scores":
        return _scores(*_indexer_inputs(case, seed), case["causal"], torch.float64)
    if op == "topk":
        s = _scores(*_indexer_inputs(case, seed), True, torch.float32)
        n_k = min(case["k_base"], K_MAX, case["T"])
        idx = torch.empty(*s.shape[:2], n_k, device="cuda", dtype=torch.int64)
        mask = torch.empty(*s.shape[:2], n_k, device="cuda", dtype=torch.bool)
        for b in range(case["B"]):
            for r0 in range(0, case["T"], 2048):
                rows = s[b, r0:r0 + 2048]
                idx[b, r0:r0 + 2048] = rows.sort(dim=-1, descending=True, stable=True).indices[:, :n_k]
                mask[b, r0:r0 + 2048] = rows.gather(1, idx[b, r0:r0 + 2048]) > -math.inf
        return idx, mask, n_k
    q, k, cos, sin = (t.double() for t in _rope_inputs(case, seed))
    return tuple(torch.stack([_rope64(t[b], cos[0, :, 0], sin[0, :, 0]) for b in range(case["B"])]) for t in (q, k))
