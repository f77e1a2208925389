"""The head_dim 64 bf16 kernels at the edges of their 32-row tiles, their wave
splits and their 64-row form, against the float64 dense oracle (bf16 bar 2e-2
norm-relative, statistics 1e-4, as the other bf16 kernels)."""

import numpy as np
import pytest

from oracle import dense
from tests.conftest import bf16_round, norm_rel

pytestmark = pytest.mark.gpu

CASES = [
    # b, nq, nk, hq, hkv, q_pos0, k_pos0, causal, valid
    (1, 1, 1, 1, 1, 0, 0, True, None),             # smallest
    (1, 31, 33, 2, 1, 5, 0, True, None),           # partial tiles either side
    (2, 32, 64, 3, 3, 32, 0, True, None),          # whole tiles, diagonal at a tile edge
    (1, 33, 32, 4, 2, 0, 0, True, None),           # a one-row query block
    (1, 65, 130, 2, 2, 70, 10, True, 100),         # offsets, valid_length inside a tile
    (1, 40, 96, 2, 1, 0, 60, True, None),          # no query sees a key
    (1, 64, 64, 1, 1, 0, 32, True, None),          # half the queries see none
    (1, 70, 90, 2, 1, 0, 0, False, None),          # non-causal
    (1, 64, 1024, 9, 3, 960, 0, True, None),       # eight key splits
    (1, 1000, 64, 6, 1, 0, 0, True, 50),           # dK/dV: eight splits over a group of six
    (64, 20, 70, 64, 16, 50, 0, True, None),       # one row block per head: four waves on its keys
    (32, 50, 70, 64, 16, 20, 0, True, 65),         # two (64-row waves for 2,048 heads): ragged
    (8, 100, 64, 16, 16, 0, 0, False, None),       # more waves than tiles
    (2, 2100, 300, 40, 20, 100, 0, True, None),    # 64-row waves with key splits
    (1, 1100, 2200, 128, 128, 1100, 0, True, 2150),  # 64-row waves, ragged tail block
]


@pytest.mark.parametrize("case", CASES)
def test_attn64_edges(gpu, case):
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, qp, kp, causal, valid = case
    rng = np.random.default_rng(nq * 31 + nk)
    q, k, v, do = (bf16_round(rng.standard_normal(s, dtype=np.float32))
                   for s in ((b, nq, hq, 64), (b, nk, hkv, 64), (b, nk, hkv, 64), (b, nq, hq, 64)))
    qt, kt, vt, dt = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in (q, k, v, do))
    kw = dict(q_pos0=qp, k_pos0=kp, causal=causal, valid_length=valid)
    o, m, l = ra.fwd_shard(qt, kt, vt, **kw)
    # a few heads of a large case are enough for the float64 oracle
    heads = sorted({0, hq - 1, hq // 2})
    kv = [h // (hq // hkv) for h in heads]
    eo, em, el = dense.attention_fwd(q[:, :, heads], k[:, :, kv], v[:, :, kv], **kw)
    o_, m_, l_ = o.cpu().numpy(), m.cpu().numpy()[:, heads], l.cpu().numpy()[:, heads]
    fin = np.isfinite(em)
    assert np.array_equal(np.isfinite(m_), fin) and np.all(l_[~fin] == 0)
    assert np.all(o_[:, :, heads][~fin.transpose(0, 2, 1)] == 0)
    if fin.any():
        assert norm_rel(o_[:, :, heads], eo) <= 2e-2 and norm_rel(l_, el) <= 1e-4
        assert np.abs(m_[fin] - em[fin]).max() <= 1e-4 * max(1.0, np.abs(em[fin]).max())
    # the epilogue's merge of the same hop into itself keeps o and doubles l
    o2, m2, l2 = o.clone(), m.clone(), l.clone()
    ra.fwd_shard(qt, kt, vt, o=o2, m=m2, l=l2, accumulate=True, **kw)
    assert gpu.equal(m2, m) and norm_rel(l2.cpu(), 2 * l.cpu()) <= 1e-6
    assert norm_rel(o2.cpu(), o.cpu()) <= 1e-6

    out = o.to(gpu.bfloat16)
    delta, lse2 = ra.bwd_preprocess(out, dt, m, l)
    acc = [gpu.zeros(x.shape, dtype=gpu.float32, device="cuda") for x in (qt, kt, vt)]
    for _ in range(2):  # the accumulators are added to
        ra.bwd_shard(qt, kt, vt, dt, lse2, delta, dq_acc=acc[0], dk_acc=acc[1], dv_acc=acc[2], **kw)
    got = [x.cpu().numpy() / 2 for x in acc]
    group = hq // hkv
    on = out.float().cpu().numpy()
    for hk in sorted({0, hkv - 1}):
        hs = slice(hk * group, (hk + 1) * group)
        ks = slice(hk, hk + 1)
        want = dense.attention_bwd(q[:, :, hs], k[:, :, ks], v[:, :, ks], do[:, :, hs],
                                   out=on[:, :, hs], **kw)
        for g, e, s in zip(got, want, (hs, ks, ks)):
            if np.abs(e).max() < 1e-3:  # one visible key: the exact gradient is rounding of out
                assert np.abs(g[:, :, s] - e).max() <= 2e-2
            else:
                assert norm_rel(g[:, :, s], e) <= 2e-2


def _rounded_p_error(q, k, v, split):
    """Distance from float64 (2-norm, relative) of an output whose only rounding
    is that of the probabilities to bf16, each relative to the exact maximum of
    the 32-key tiles so far, the tiles dealt to `split` partial results that are
    merged exactly: what the kernel's arithmetic leaves at best."""
    s = (q @ k.T) * q.shape[1] ** -0.5
    p = np.exp(s - s.max(1, keepdims=True))
    exact = (p @ v) / p.sum(1, keepdims=True)
    parts = []
    for i in range(split):
        m = np.full((len(q), 1), -np.inf)
        acc, l = np.zeros_like(exact), np.zeros((len(q), 1))
        for t in range(i * 32, len(k), 32 * split):
            x = s[:, t:t + 32]
            m_new = np.maximum(m, x.max(1, keepdims=True))
            p = np.exp(x - m_new)
            f = np.exp(m - m_new)
            acc = acc * f + bf16_round(p.astype(np.float32)).astype(np.float64) @ v[t:t + 32]
            l, m = l * f + p.sum(1, keepdims=True), m_new
        parts.append((m, acc, l))
    top = np.max([m for m, _, _ in parts], axis=0)
    num = sum(a * np.exp(m - top) for m, a, _ in parts)
    den = sum(x * np.exp(m - top) for m, _, x in parts)
    return norm_rel(num / den, exact)


@pytest.mark.parametrize("nq,nk,h", [(64, 513, 1), (33, 300, 3), (200, 1000, 40)])
def test_forward_probabilities_relative_to_the_exact_maximum(gpu, nq, nk, h):
    """The fp32 output is no further from float64 than rounding the
    probabilities against each tile's running maximum leaves it (1% for the
    hardware exponential's last bit).  Against a maximum that may lag behind by
    a factor of 2^8 no probability is an exact power of two and the distance
    grows by 5-15%."""
    from longctx100m_amd import ring_attention as ra

    rng = np.random.default_rng(nq + nk)
    q, k, v = (bf16_round(rng.standard_normal((2, n, h, 64), dtype=np.float32))
               for n in (nq, nk, nk))
    o, _, l = ra.fwd_shard(*(gpu.tensor(x).to(gpu.bfloat16).cuda() for x in (q, k, v)),
                           q_pos0=0, k_pos0=0, causal=False)
    f = [x.astype(np.float64) for x in (q, k, v)]
    heads = sorted({0, h // 2, h - 1})
    got, lim = [], []
    for b in range(2):
        for i in heads:
            args = [x[b, :, i] for x in f]
            s = args[0] @ args[1].T / 8
            p = np.exp(s - s.max(1, keepdims=True))
            got.append(norm_rel(o[b, :, i].cpu().numpy(), p @ args[2] / p.sum(1, keepdims=True)))
            assert norm_rel(l[b, i].cpu().numpy(), p.sum(1)) <= 1e-6
            lim.append(max(_rounded_p_error(*args, split) for split in (1, 8)))
    assert np.mean(got) <= 1.01 * np.mean(lim), (got, lim)
