"""The fp32-math kernels (any head_dim, fp32 or bf16 inputs on the fp32 matrix
cores) at the edges of their tiles, head-dim blocks and workgroup splits,
against the float64 dense oracle."""

import numpy as np
import pytest

from oracle import dense
from tests.conftest import bf16_round, norm_rel

pytestmark = pytest.mark.gpu

# Sums of up to 4,096 fp32 terms in another order: the bar of the fp32 path.
TOL = 1e-5

CASES = [
    # b, nq, nk, hq, hkv, d, q_pos0, k_pos0, causal, valid, dtype, element offset of every base
    (1, 1, 1, 1, 1, 1, 0, 0, False, None, "float32", 0),     # smallest; dims below one block
    (1, 15, 33, 2, 1, 16, 20, 0, True, None, "float32", 0),  # partial tiles, one dim block
    (2, 17, 16, 3, 3, 20, 0, 0, True, None, "float32", 1),   # unaligned rows: single elements
    (1, 64, 65, 4, 2, 33, 10, 3, True, 60, "float32", 0),    # odd head_dim
    (1, 100, 130, 6, 2, 96, 40, 0, True, None, "bfloat16", 0),   # six dim blocks (8-byte vectors)
    (1, 100, 130, 6, 2, 90, 40, 0, True, None, "bfloat16", 0),   # the same, head_dim % 4 != 0
    (1, 48, 200, 2, 1, 128, 200, 0, True, 190, "float32", 0),    # K and V fragments in LDS
    (1, 33, 70, 2, 2, 100, 0, 0, False, None, "bfloat16", 3),    # eight blocks, unaligned
    (1, 40, 90, 2, 1, 192, 60, 0, True, None, "float32", 0),     # sixteen blocks, four waves
    (1, 31, 47, 1, 1, 256, 0, 16, True, None, "float32", 0),     # queries before the first key
    (1, 16, 1100, 9, 3, 64, 1084, 0, True, None, "float32", 0),  # eight key splits
    (1, 700, 600, 9, 3, 64, 0, 0, True, 555, "float32", 0),      # splits, causal from the start
    (2, 1030, 40, 33, 11, 32, 900, 870, True, None, "float32", 0),  # two query blocks per wave
]


def _offset(torch, arr, dtype, off):
    """A contiguous device tensor of arr whose base is off elements past an aligned one."""
    t = torch.zeros(arr.size + off, dtype=dtype, device="cuda")
    t[off:] = torch.tensor(arr.reshape(-1), dtype=torch.float32).to(dtype).cuda()
    return t[off:].view(arr.shape)


@pytest.mark.parametrize("case", CASES)
def test_fp32_math_edges(gpu, case):
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, d, qp, kp, causal, valid, dt, off = case
    rng = np.random.default_rng(nq * 1000 + nk + d)
    dtype = getattr(gpu, dt)
    arrs = [rng.standard_normal(s).astype(np.float32)
            for s in ((b, nq, hq, d), (b, nk, hkv, d), (b, nk, hkv, d), (b, nq, hq, d))]
    if dt == "bfloat16":
        arrs = [bf16_round(x) for x in arrs]
    q, k, v, do = (_offset(gpu, x, dtype, off) for x in arrs)
    kw = dict(q_pos0=qp, k_pos0=kp, causal=causal, valid_length=valid)
    o, m, l = ra.fwd_shard(q, k, v, precise=True, **kw)
    eo, em, el = dense.attention_fwd(*arrs[:3], **kw)
    o_, m_, l_ = (t.cpu().numpy() for t in (o, m, l))
    fin = np.isfinite(em)
    assert np.array_equal(np.isfinite(m_), fin) and np.all(l_[~fin] == 0)
    assert np.all(o_[~fin.transpose(0, 2, 1)] == 0)
    assert norm_rel(o_, eo) <= TOL and norm_rel(l_, el) <= TOL
    assert np.abs(m_[fin] - em[fin]).max() <= TOL * max(1.0, np.abs(em[fin]).max())
    # the epilogue's merge of the same hop into itself keeps o and doubles l
    ra.fwd_shard(q, k, v, precise=True, o=o, m=m, l=l, accumulate=True, **kw)
    assert norm_rel(o.cpu().numpy(), eo) <= TOL and norm_rel(l.cpu().numpy(), 2 * el) <= TOL

    # backward from the oracle's statistics; accumulators start at one
    out = _offset(gpu, eo.astype(np.float32), dtype, off)
    mm, ll = (gpu.tensor(x, dtype=gpu.float32).contiguous().cuda() for x in (em, el))
    delta, lse2 = ra.bwd_preprocess(out, do, mm, ll)
    acc = [gpu.ones(x.shape, dtype=gpu.float32, device="cuda") for x in (q, k, v)]
    ra.bwd_shard(q, k, v, do, lse2, delta, precise=True, dq_acc=acc[0], dk_acc=acc[1],
                 dv_acc=acc[2], **kw)
    want = dense.attention_bwd(*arrs, out=out.float().cpu().numpy(), **kw)
    for got, e in zip(acc, want):
        # the sum with the starting one rounds at one ulp of a number of the gradient's size plus one
        assert np.abs(got.cpu().numpy() - 1 - e).max() <= TOL * (1 + np.abs(e).max())


def _fma(a, b, c):
    """fp32 fused multiply-add: the product of two fp32 values is exact in float64."""
    return (a.double() * b.double() + c.double()).float()


@pytest.mark.parametrize("d", [64, 96, 128])
def test_scores_as_exact_as_four_lane_dot_products(gpu, d):
    """The rounding of the scores, seen in the row maxima: on average no larger
    than that of plain fp32 dot products of four chains of d / 4 fused
    multiply-adds.  (10%: three standard deviations of the mean of 2,000
    errors; two chains of twice the length are 1.4 times as far off.)"""
    from longctx100m_amd import ring_attention as ra

    n, heads = 1000, 32
    g = gpu.Generator().manual_seed(d)
    q, k, v = (gpu.randn(2, n, h, d, generator=g) for h in (heads, 8, 8))
    _, m, _ = ra.fwd_shard(*(x.cuda() for x in (q, k, v)), q_pos0=0, k_pos0=0, causal=False)
    got = lim = 0.0
    for h in (0, 31):
        qh, kh = q[0, :, h], k[0, :, h // 4]
        exact = (qh.double() @ kh.double().T * d ** -0.5).max(1).values
        part = [gpu.zeros(n, n) for _ in range(4)]
        for j in range(0, d, 4):
            for e in range(4):
                part[e] = _fma(qh[:, j + e, None], kh[None, :, j + e], part[e])
        s = ((part[0] + part[1]) + (part[2] + part[3])) * gpu.tensor(d ** -0.5).float()
        lim += float((s.max(1).values.double() - exact).abs().mean())
        got += float((m[0, h].cpu().double() - exact).abs().mean())
    assert got <= 1.1 * lim, (got, lim)
