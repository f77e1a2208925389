"""The work a user of this package gives it, as measurable cases.

Every case goes through a public entry point of longctx100m_amd: the ring's
reference signatures (forward with statistics, two-pass backward), one rank's
step with per-owner dK/dV, a prompt chunk against a KV cache, split-KV decode,
and a decoder layer's prefill and decode.  Kinds and what they stand for:

  train     the attention of a training step: forward of every rank of the
            in-process ring, then one rank's backward (world 1 is dense
            attention, the call a model without a ring makes)
  rank      one rank's share of a ring with resident KV shards: forward, then
            dQ and the per-owner dK/dV it sends back
  prefill   one rank's forward over its own and the preceding KV shards
  chunk     a prompt chunk of a few hundred tokens against the keys before it
            (chunked prefill)
  decode    one to eight new tokens per sequence against a KV cache
            (several tokens: a verified draft)
  layer_prefill, layer_decode
            a whole decoder layer (norms, projections, RoPE, attention,
            SwiGLU) over a prompt, and for one new token
"""

from __future__ import annotations

import math

import torch

from longctx100m_amd import layer as L
from longctx100m_amd import rank_step as rs
from longctx100m_amd import ring_attention as ra

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # One new token, short context: the smallest call, launches and latency.
        dict(name="decode_short", kind="decode", batch=1, tokens=1, cache=500, hq=32, hkv=8, d=128,
             dtype="bf16"),
        # One new token over a 262,144-token cache of a GQA 32/8 layer.
        dict(name="decode_long", kind="decode", batch=1, tokens=1, cache=262144, hq=32, hkv=8,
             d=128, dtype="bf16"),
        # A batch of conversations of a small GQA 9/3, head_dim 64 model, ragged length.
        dict(name="decode_batch_d64", kind="decode", batch=4, tokens=1, cache=3001, hq=9, hkv=3,
             d=64, dtype="bf16"),
        # Eight drafted tokens checked at once against a 16k context.
        dict(name="decode_draft", kind="decode", batch=1, tokens=8, cache=16001, hq=32, hkv=8,
             d=128, dtype="bf16"),
        # The two-rank fp32 ring of the parity setup, forward and backward.
        dict(name="train_fp32_ring", kind="train", world=2, rank=1, batch=1, n=512, hq=9, hkv=3,
             d=64, dtype="fp32", valid=0),
        # bf16 training attention of the same heads on ragged sequences, dense.
        dict(name="train_bf16_d64", kind="train", world=1, rank=0, batch=2, n=2047, hq=9, hkv=3,
             d=64, dtype="bf16", valid=0),
        # bf16 training attention of a GQA 32/8 layer at an ordinary context length, padded.
        dict(name="train_bf16_gqa", kind="train", world=1, rank=0, batch=1, n=4096, hq=32, hkv=8,
             d=128, dtype="bf16", valid=4000),
        # The 32,768-token bf16 shard of 16 heads: diagonal and one preceding shard, the largest.
        dict(name="rank_step_32k", kind="rank", world=2, rank=1, batch=1, n=32768, hq=16, hkv=16,
             d=128, dtype="bf16"),
        # A prefill share: the last of four 8,192-token shards of a GQA 32/8 layer.
        dict(name="prefill_ring_gqa", kind="prefill", world=4, rank=3, batch=1, n=8192, hq=32,
             hkv=8, d=128, dtype="bf16"),
        # Chunked prefill: 512 prompt tokens against 32k earlier ones and themselves.
        dict(name="chunk_512_32k", kind="chunk", batch=1, tokens=512, past=32000, hq=32, hkv=8,
             d=128, dtype="bf16"),
        # A decoder layer (hidden 4096, GQA 32/8, SwiGLU 14336) over a 2,000-token prompt.
        dict(name="layer_prefill_2k", kind="layer_prefill", tokens=2000),
        # The same layer for one new token at position 8,000.
        dict(name="layer_decode_8k", kind="layer_decode", pos=8000),
    ]


HEADS = ((9, 3), (16, 16), (32, 8), (8, 2))


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over the logarithm, odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("train", "train", "train", "rank", "prefill", "chunk", "decode", "decode",
                       "decode", "layer_prefill", "layer_decode"))
    hq, hkv = rng.choice(HEADS)
    if kind == "train":
        dtype = rng.choice(("fp32", "bf16", "bf16"))
        d = rng.choice((64, 128, 128, 96))
        world = rng.choice((1, 1, 2, 3))
        # head_dim 96 and fp32 inputs take the fp32-math kernels
        n = _log(rng, 33, 1000 if dtype == "fp32" or d == 96 else 4096)
        valid = rng.choice((0, 0, max(1, world * n - rng.randrange(1, n))))
        return dict(kind=kind, world=world, rank=rng.randrange(world), batch=rng.choice((1, 2)),
                    n=n, hq=hq, hkv=hkv, d=d, dtype=dtype, valid=valid)
    if kind == "rank":
        world = rng.choice((1, 2, 3))
        return dict(kind=kind, world=world, rank=world - 1, batch=1, n=_log(rng, 500, 8192), hq=hq,
                    hkv=hkv, d=128, dtype="bf16")
    if kind == "prefill":
        world = rng.choice((1, 2, 3, 4))
        return dict(kind=kind, world=world, rank=rng.randrange(world), batch=1,
                    n=_log(rng, 200, 8192), hq=hq, hkv=hkv, d=rng.choice((64, 128)), dtype="bf16")
    if kind == "chunk":
        return dict(kind=kind, batch=1, tokens=_log(rng, 17, 2048), past=_log(rng, 500, 60000),
                    hq=hq, hkv=hkv, d=rng.choice((64, 128, 128)), dtype="bf16")
    if kind == "decode":
        return dict(kind=kind, batch=rng.choice((1, 2, 4, 7, 16)), tokens=rng.choice((1, 1, 2, 5, 8)),
                    cache=_log(rng, 65, 60000), hq=hq, hkv=hkv, d=rng.choice((64, 128, 128)),
                    dtype="bf16")
    if kind == "layer_prefill":
        return dict(kind=kind, tokens=_log(rng, 33, 4096))
    return dict(kind=kind, pos=_log(rng, 33, 60000))


# ------------------------------------------------------------------ inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _qkv(case, g, nq, nk):
    """N(0,1) queries, keys and values, as after a normalised projection."""
    dt, b, d = DTYPES[case["dtype"]], case["batch"], case["d"]
    return (_randn(g, b, nq, case["hq"], d, dtype=dt), _randn(g, b, nk, case["hkv"], d, dtype=dt),
            _randn(g, b, nk, case["hkv"], d, dtype=dt))


def _shards(case, g):
    return [_qkv(case, g, case["n"], case["n"]) for _ in range(case["world"])]


def _grads(case, g, count):
    dt = DTYPES[case["dtype"]]
    return [_randn(g, case["batch"], case["n"], case["hq"], case["d"], dtype=dt)
            for _ in range(count)]


def _layer_inputs(case, g):
    cfg = L.C4
    w = L.init_layer_weights(cfg, g, DEV)
    for name in ("norm1", "norm2"):  # trained norms are near one, not at it
        w[name] = (1 + 0.1 * _randn(g, cfg.hidden_size, dtype=torch.float32)).to(torch.bfloat16)
    n = case["tokens"] if case["kind"] == "layer_prefill" else 1
    x = _randn(g, n, cfg.hidden_size)
    res = _randn(g, n, cfg.hidden_size)  # the previous layer's MLP output, still to be added
    return cfg, w, x, res


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "train":
        st["shards"] = _shards(case, g)
        st["grads"] = _grads(case, g, case["world"])
    elif kind == "rank":
        shards = _shards(case, g)
        dout, = _grads(case, g, 1)
        st["step"] = rs.RankStep(shards[case["rank"]][0], dout, [s[1] for s in shards],
                                 [s[2] for s in shards], case["rank"])
    elif kind == "prefill":
        st["shards"] = _shards(case, g)
    elif kind == "chunk":
        st["qkv"] = _qkv(case, g, case["tokens"], case["past"] + case["tokens"])
    elif kind == "decode":
        st["qkv"] = q, k, _ = _qkv(case, g, case["tokens"], case["cache"])
        # a serving loop keeps the scratch of its decode calls
        sh = ra._shape(q, k, False)
        need = ra._lib.load().lc_attn_decode_workspace_bytes(sh)
        st["ws"] = torch.empty(max(1, need), dtype=torch.uint8, device=DEV)
    elif kind == "layer_prefill":
        cfg, w, x, res = _layer_inputs(case, g)
        rope = L.rope_params(cfg.head_dim, cfg.rope_theta, cfg.rope_scaling)
        st.update(cfg=cfg, w=w, x=x, res=res, table=L.rope_table(rope, case["tokens"], 0))
    else:
        cfg, w, x, res = _layer_inputs(case, g)
        pos = case["pos"]
        rope = L.rope_params(cfg.head_dim, cfg.rope_theta, cfg.rope_scaling)
        shape = (1, pos + 1, cfg.num_key_value_heads, cfg.head_dim)
        sh = ra._lib.Shape(1, 1, pos + 1, cfg.num_heads, cfg.num_key_value_heads, cfg.head_dim,
                           ra._lib.LC_DTYPE_BF16, 0)
        need = ra._lib.load().lc_attn_decode_workspace_bytes(sh)
        st.update(cfg=cfg, w=w, x=x, res=res, table=L.rope_table(rope, pos + 1, 0),
                  cache=(_randn(g, *shape), _randn(g, *shape)),
                  ws=torch.empty(max(1, need), dtype=torch.uint8, device=DEV))
    return st


# ---------------------------------------------------------------- one pass --

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        shards, r = state["shards"], case["rank"]
        valid = case["valid"] or None
        fwd = [ra.ring_causal_attention_forward_with_stats(shards, i, valid_length=valid)
               for i in range(case["world"])]
        outs, ms, ls = (list(x) for x in zip(*fwd))
        dq, dk, dv = ra.ring_causal_attention_backward(shards, r, outs, ms, ls, state["grads"],
                                                       valid_length=valid)
        return {"out": outs[r], "m": ms[r], "l": ls[r], "dq": dq, "dk": dk, "dv": dv}
    if kind == "rank":
        step = state["step"]
        step.step()
        return {"out": step.out, "m": step.m, "l": step.l, "dq": step.dq_acc,
                "dk": [step.dk_acc[o] for o in step.owners],
                "dv": [step.dv_acc[o] for o in step.owners]}
    if kind == "prefill":
        out, m, l = ra.ring_causal_attention_forward_with_stats(state["shards"], case["rank"])
        return {"out": out, "m": m, "l": l}
    if kind == "chunk":
        q, k, v = state["qkv"]
        o, m, l = ra.fwd_shard(q, k, v, q_pos0=case["past"], k_pos0=0)
        return {"out": o, "m": m, "l": l}
    if kind == "decode":
        q, k, v = state["qkv"]
        o, m, l = ra.decode(q, k, v, q_pos0=case["cache"] - case["tokens"], workspace=state["ws"])
        return {"out": o, "m": m, "l": l}
    if kind == "layer_prefill":
        x, mlp = L.layer_prefill(state["x"], state["w"], state["cfg"], state["table"], 0, [],
                                 residual=state["res"])
        return {"x": x, "mlp": mlp}
    cache, pos = state["cache"], case["pos"]
    x, mlp = L.layer_decode(state["x"], state["w"], state["cfg"], state["table"], pos, cache,
                            residual=state["res"], workspace=state["ws"])
    return {"x": x, "mlp": mlp, "k": cache[0][:, pos], "v": cache[1][:, pos]}


# -------------------------------------------------------------------- work --

def _pairs(nq, nk, q0, valid):
    """Visible (query, key) pairs of queries q0 .. q0+nq-1 over keys 0 .. nk-1."""
    nk = min(nk, valid) if valid else nk
    full = max(0, min(nq, q0 + nq - nk + 1))  # queries that see all nk keys
    part = nq - full
    return full * nk + part * q0 + part * (part + 1) // 2


def _hop_pairs(case, qr, kr):
    """Visible pairs of rank qr's queries and rank kr's keys."""
    n, valid = case["n"], case.get("valid", 0)
    hi = _pairs(n, (kr + 1) * n, qr * n, valid)
    return hi - (_pairs(n, kr * n, qr * n, valid) if kr else 0)


def _layer_work(cfg, tokens):
    d, hq, hkv, c, inter = (cfg.head_dim, cfg.num_heads, cfg.num_key_value_heads, cfg.hidden_size,
                            cfg.intermediate_size)
    weights = c * ((hq + 2 * hkv) * d + hq * d + 3 * inter)
    return {"bytes": 2 * weights + 2 * tokens * c * 4, "flops": 2 * tokens * weights}


def work(case):
    kind = case["kind"]
    if kind == "layer_prefill":
        w, t = _layer_work(L.C4, case["tokens"]), case["tokens"]
        w["flops"] += 4 * _pairs(t, t, 0, 0) * L.C4.num_heads * L.C4.head_dim
        return w
    if kind == "layer_decode":
        w, n = _layer_work(L.C4, 1), case["pos"] + 1
        w["bytes"] += 4 * n * L.C4.num_key_value_heads * L.C4.head_dim
        w["flops"] += 4 * n * L.C4.num_heads * L.C4.head_dim
        return w
    b, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["d"]
    es = 4 if case["dtype"] == "fp32" else 2
    unit = 4 * b * hq * d  # flops of a visible pair, forward; the backward is 2.5 times that
    if kind in ("chunk", "decode"):
        nq = case["tokens"]
        nk = case["cache"] if kind == "decode" else case["past"] + nq
        return {"bytes": b * (nq * hq * d * (es + 4) + 2 * nk * hkv * d * es + 8 * nq * hq),
                "flops": unit * _pairs(nq, nk, nk - nq, 0)}
    n, w, r = case["n"], case["world"], case["rank"]
    qn, kn, sn = b * n * hq * d, b * n * hkv * d, b * n * hq
    if kind == "prefill":
        return {"bytes": 2 * qn * es + 2 * (r + 1) * kn * es + 8 * sn,
                "flops": unit * sum(_hop_pairs(case, r, k) for k in range(r + 1))}
    if kind == "rank":
        pairs = sum(_hop_pairs(case, r, k) for k in range(r + 1))
        return {"bytes": 3 * qn * es + 4 * qn + (r + 1) * kn * (2 * es + 8) + 8 * sn,
                "flops": 3.5 * unit * pairs}
    fwd = sum(_hop_pairs(case, q, k) for q in range(w) for k in range(q + 1))
    # the backward's two passes: dK/dV (4 products) of this rank's keys over every query owner,
    # dQ (1 product more, 3 where the pair is not this rank's own) over every KV owner
    own = _hop_pairs(case, r, r)
    bwd = 2.5 * own + 2 * sum(_hop_pairs(case, q, r) for q in range(r + 1, w)) \
        + 1.5 * sum(_hop_pairs(case, r, k) for k in range(r))
    return {"bytes": w * (qn * es * 3 + 2 * kn * es + 8 * sn) + (qn + 2 * kn) * es,
            "flops": unit * (fwd + bwd)}


# --------------------------------------------------------------- tolerance --

def tolerance(case):
    """About four times the distance between two correct implementations at
    the case's precision: fp32 sums in another order (measured 2e-7 to 1e-6 of
    the 2-norm), bf16 probabilities and outputs (2e-3 to 3e-3 from the exact
    result, and 3e-3 for gradients), and for a whole layer the roundings of its
    bf16 activations on top."""
    if case["kind"] in ("layer_prefill", "layer_decode"):
        return {"rel": 2e-2}
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    return {"rel": 1e-2}


# ------------------------------------------------------------------- exact --

def _attend(q, k, v, q0, valid, group, dout=None):
    """float64 attention of q [n, Hq, d] at positions q0.. over k, v
    [m, Hkv, d]: (out, m, l) and, given dout, (dq, dk, dv)."""
    n, hq, d = q.shape
    m_ = k.shape[0]
    scale = d ** -0.5
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    mm = torch.empty(hq, n, dtype=torch.float64, device=q.device)
    ll = torch.empty_like(mm)
    dq = torch.zeros_like(out)
    dk = torch.zeros(m_, k.shape[1], d, dtype=torch.float64, device=q.device)
    dv = torch.zeros_like(dk)
    keys = torch.arange(m_, device=q.device)
    step = 4096
    for i0 in range(0, n, step):
        i1 = min(n, i0 + step)
        qpos = q0 + torch.arange(i0, i1, device=q.device)
        bad = keys[None, :] > qpos[:, None]
        if valid:
            bad |= (keys >= valid)[None, :]
        for h in range(hq):
            kh, vh = k[:, h // group].double(), v[:, h // group].double()
            qh = q[i0:i1, h].double()
            s = (qh @ kh.t()).mul_(scale).masked_fill_(bad, -math.inf)
            mx = s.max(1).values
            p = (s - mx.masked_fill(mx == -math.inf, 0)[:, None]).exp_()
            l = p.sum(1)
            p /= l.masked_fill(l == 0, 1)[:, None]
            o = p @ vh
            out[i0:i1, h], mm[h, i0:i1], ll[h, i0:i1] = o, mx, l
            if dout is not None:
                g = dout[i0:i1, h].double()
                dv[:, h // group] += p.t() @ g
                ds = p * (g @ vh.t() - (g * o).sum(1)[:, None])
                dq[i0:i1, h] = (ds @ kh) * scale
                dk[:, h // group] += (ds.t() @ qh) * scale
    return out, mm, ll, dq, dk, dv


def _exact_layer(case, seed):
    g = _gen(seed)
    cfg, w, x, res = _layer_inputs(case, g)
    w = {k: t.double() for k, t in w.items()}
    d, hq, hkv, inter = cfg.head_dim, cfg.num_heads, cfg.num_key_value_heads, cfg.intermediate_size
    pos0 = 0 if case["kind"] == "layer_prefill" else case["pos"]
    n = x.shape[0]

    def norm(h, weight):
        return h / (h.pow(2).mean(-1, keepdim=True) + cfg.rms_norm_eps).sqrt() * weight

    inv = (1.0 / cfg.rope_theta ** (torch.arange(0, d, 2, dtype=torch.float64) / d)).float().to(DEV)
    ang = ((pos0 + torch.arange(n, device=DEV)).float()[:, None] * inv).double()[:, None]

    def rope(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()), -1)

    h0 = x.double() + res.double()
    qkv = norm(h0, w["norm1"]) @ w["wqkv"].t()
    q = rope(qkv[:, :hq * d].reshape(n, hq, d))
    k = rope(qkv[:, hq * d:(hq + hkv) * d].reshape(n, hkv, d))
    v = qkv[:, (hq + hkv) * d:].reshape(n, hkv, d)
    ka, va = k, v
    if case["kind"] == "layer_decode":
        shape = (1, pos0 + 1, hkv, d)
        kc, vc = _randn(g, *shape), _randn(g, *shape)
        ka = torch.cat((kc[0, :pos0].double(), k))
        va = torch.cat((vc[0, :pos0].double(), v))
    att = _attend(q, ka, va, pos0, 0, hq // hkv)[0]
    x2 = h0 + att.reshape(n, hq * d) @ w["wo"].t()
    gu = norm(x2, w["norm2"]) @ w["wgu"].t()
    a = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    r = {"x": x2, "mlp": a @ w["wd"].t()}
    if case["kind"] == "layer_decode":
        r["k"], r["v"] = k, v
    return r


def exact(case, seed):
    kind = case["kind"]
    if kind in ("layer_prefill", "layer_decode"):
        return _exact_layer(case, seed)
    if kind == "rank" and case["n"] > 16384:
        return None
    g = _gen(seed)
    group = case["hq"] // case["hkv"]
    if kind in ("chunk", "decode"):
        nq = case["tokens"]
        nk = case["cache"] if kind == "decode" else case["past"] + nq
        q, k, v = _qkv(case, g, nq, nk)
        per = [_attend(q[i], k[i], v[i], nk - nq, 0, group) for i in range(case["batch"])]
        return {"out": torch.stack([p[0] for p in per]), "m": torch.stack([p[1] for p in per]),
                "l": torch.stack([p[2] for p in per])}
    n, w, r, valid = case["n"], case["world"], case["rank"], case.get("valid", 0)
    shards = _shards(case, g)
    out, m, l, dq, dk, dv = [], [], [], [], [], []
    grads = _grads(case, g, w if kind == "train" else 1) if kind != "prefill" else None
    for b in range(case["batch"]):
        k, v = (torch.cat([s[i][b] for s in shards]) for i in (1, 2))
        if kind == "train":  # every rank's queries act on this rank's keys
            q = torch.cat([s[0][b] for s in shards])
            o_, m_, l_, dq_, dk_, dv_ = _attend(q, k, v, 0, valid, group,
                                                torch.cat([t[b] for t in grads]))
            sl = slice(r * n, (r + 1) * n)
            o_, m_, l_, dq_, dk_, dv_ = o_[sl], m_[:, sl], l_[:, sl], dq_[sl], dk_[sl], dv_[sl]
        else:
            o_, m_, l_, dq_, dk_, dv_ = _attend(shards[r][0][b], k, v, r * n, valid, group,
                                                grads[0][b] if grads else None)
        for to, x in zip((out, m, l, dq, dk, dv), (o_, m_, l_, dq_, dk_, dv_)):
            to.append(x)
    out, m, l, dq, dk, dv = (torch.stack(x) for x in (out, m, l, dq, dk, dv))
    if kind == "rank":
        owners = [(r - h) % w for h in range(w)]
        return {"out": out, "m": m, "l": l, "dq": dq,
                "dk": [dk[:, o * n:(o + 1) * n] for o in owners],
                "dv": [dv[:, o * n:(o + 1) * n] for o in owners]}
    stats = {"out": out, "m": m[..., None], "l": l[..., None]}
    return stats if kind == "prefill" else dict(stats, dq=dq, dk=dk, dv=dv)
