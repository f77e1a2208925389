"""The head_dim 128 forward with its keys split over the chip (small grids with
a workspace), against the float64 dense oracle and the unsplit call (bf16 bar
2e-2 norm-relative, statistics 1e-4)."""

import ctypes

import numpy as np
import pytest

from longctx100m_amd import _lib
from oracle import dense
from tests.conftest import bf16_round, norm_rel

CASES = [
    # b, nq, nk, hq, hkv, q_pos0, k_pos0, causal, valid
    (1, 1, 1024, 1, 1, 1023, 0, True, None),       # two splits
    (1, 33, 1600, 2, 1, 1567, 0, True, None),      # three, ragged last split
    (1, 129, 8200, 8, 2, 8071, 0, True, None),     # sixteen, two query tiles
    (2, 40, 3000, 4, 4, 3000, 0, True, None),      # no diagonal: eight-wave workgroups
    (1, 64, 4096, 2, 2, 4032, 0, True, 1100),      # valid_length: later splits see no key
    (1, 200, 2100, 2, 1, 0, 0, True, None),        # causal from the start: splits without keys
    (1, 50, 2000, 2, 2, 30, 60, True, None),       # rows before every key
    (1, 70, 5000, 3, 1, 0, 0, False, None),        # non-causal
]


def _bytes(lib, shape):
    return lib.lc_attn_fwd_shard_workspace_bytes(ctypes.byref(shape))


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_fwd_splits(gpu, case):
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, qp, kp, causal, valid = case
    rng = np.random.default_rng(nq + nk)
    q, k, v = (bf16_round(rng.standard_normal(s, dtype=np.float32))
               for s in ((b, nq, hq, 128), (b, nk, hkv, 128), (b, nk, hkv, 128)))
    qt, kt, vt = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in (q, k, v))
    kw = dict(q_pos0=qp, k_pos0=kp, causal=causal, valid_length=valid)
    lib = _lib.load()
    s = _lib.Shape(b, nq, nk, hq, hkv, 128, _lib.LC_DTYPE_BF16, 0)
    assert _bytes(lib, s) > 0
    o, m, l = ra.fwd_shard(qt, kt, vt, **kw)
    eo, em, el = dense.attention_fwd(q, k, v, **kw)
    fin = np.isfinite(em)
    o_, m_, l_ = (t.cpu().numpy() for t in (o, m, l))
    assert np.array_equal(np.isfinite(m_), fin) and np.all(l_[~fin] == 0)
    assert np.all(o_[~fin.transpose(0, 2, 1)] == 0)
    assert norm_rel(o_, eo) <= 2e-2 and norm_rel(l_, el) <= 1e-4
    assert np.abs(m_[fin] - em[fin]).max() <= 1e-4 * max(1.0, np.abs(em[fin]).max())

    # the entry without a workspace: the same up to rounding
    mk = _lib.Mask(qp, kp, -1 if valid is None else valid, int(causal), 0)
    o1, m1, l1 = (gpu.full_like(t, float("nan")) for t in (o, m, l))
    _lib.check(lib.lc_attn_fwd_shard(s, mk, *(t.data_ptr() for t in (qt, kt, vt, o1, m1, l1)),
                                     gpu.cuda.current_stream().cuda_stream))
    assert gpu.equal(m, m1) and norm_rel(l.cpu(), l1.cpu()) <= 1e-5
    assert norm_rel(o.cpu(), o1.cpu()) <= 1e-2  # bf16 probabilities relative to other maxima

    # merged into itself the hop keeps o and m and doubles l
    ra.fwd_shard(qt, kt, vt, o=o, m=m, l=l, accumulate=True, **kw)
    assert np.array_equal(m.cpu().numpy(), m_) and norm_rel(l.cpu().numpy(), 2 * l_) <= 1e-6
    assert norm_rel(o.cpu().numpy(), o_) <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["query", "key"])
def test_nan_passes_through_the_splits(gpu, where):
    """A NaN query leaves every split of its row without a maximum: the row is
    NaN as in the unsplit call, not zeros; a NaN key reaches the rows that see it."""
    from longctx100m_amd import ring_attention as ra

    nq, nk = 33, 2100
    q, k, v = (gpu.randn(1, n, 2, 128, device="cuda").to(gpu.bfloat16) for n in (nq, nk, nk))
    if where == "query":
        q[0, 7, 1] = float("nan")
    else:
        k[0, 2090, 1, 5] = float("nan")
    mk = _lib.Mask(nk - nq, 0, -1, 1, 0)
    o, m, l = ra.fwd_shard(q, k, v, q_pos0=nk - nq, k_pos0=0)
    o1, m1, l1 = (gpu.zeros_like(t) for t in (o, m, l))
    _lib.check(_lib.load().lc_attn_fwd_shard(
        _lib.Shape(1, nq, nk, 2, 2, 128, _lib.LC_DTYPE_BF16, 0), mk,
        *(t.data_ptr() for t in (q, k, v, o1, m1, l1)), gpu.cuda.current_stream().cuda_stream))
    want = gpu.zeros(nq, 2, dtype=gpu.bool)
    if where == "query":
        want[7, 1] = True
    else:
        want[2090 - (nk - nq):, 1] = True
    for t in (o, o1):
        assert gpu.equal(t[0].isnan().all(-1).cpu(), want)
        assert gpu.equal(t[0].isnan().any(-1).cpu(), want)


@pytest.mark.gpu
def test_ring_forward_with_the_least_workspace(gpu):
    """lc_ring_fwd_with_stats takes the running output alone as its workspace and
    then runs its hops unsplit."""
    rng = np.random.default_rng(5)
    world, n, hq, hkv, d = 2, 1100, 4, 2, 128
    mk = lambda h: gpu.tensor(rng.standard_normal((1, n, h, d)),  # noqa: E731
                              dtype=gpu.float32).to(gpu.bfloat16).cuda()
    qs, ks, vs = ([mk(h) for _ in range(world)] for h in (hq, hkv, hkv))
    lib = _lib.load()
    desc = _lib.RingDesc(world, 1, 1, n, hq, hkv, d, _lib.LC_DTYPE_BF16, 0, 1, 64, 128, -1, -1)
    least = -(-n * hq * d * 4 // 256) * 256
    full = lib.lc_ring_fwd_workspace_bytes(desc)
    assert full > least
    res = []
    for nbytes in (least, full):
        ws = gpu.empty(nbytes, dtype=gpu.uint8, device="cuda")
        out = gpu.empty_like(qs[1])
        m, l = (gpu.empty((1, hq, n), device="cuda") for _ in range(2))
        arrs = [_lib.ptr_array([t.data_ptr() for t in ts]) for ts in (qs, ks, vs)]
        _lib.check(lib.lc_ring_fwd_with_stats(desc, *(a[0] for a in arrs), out.data_ptr(),
                                              m.data_ptr(), l.data_ptr(), ws.data_ptr(), nbytes,
                                              gpu.cuda.current_stream().cuda_stream))
        res.append((out.float().cpu(), m.cpu(), l.cpu()))
    assert gpu.equal(res[0][1], res[1][1])
    assert norm_rel(res[0][0], res[1][0]) <= 1e-2 and norm_rel(res[0][2], res[1][2]) <= 1e-5
    assert lib.lc_ring_fwd_with_stats(desc, *(a[0] for a in arrs), out.data_ptr(), m.data_ptr(),
                                      l.data_ptr(), ws.data_ptr(), least - 256,
                                      None) == _lib.LC_ERR_WORKSPACE


def test_split_workspace_sizes():
    lib = _lib.load()
    sh = lambda b, nq, nk, hq, hkv, d, dt, fl=0: _lib.Shape(b, nq, nk, hq, hkv, d, dt, fl)  # noqa: E731
    bf, f32 = _lib.LC_DTYPE_BF16, _lib.LC_DTYPE_F32
    assert _bytes(lib, sh(1, 512, 32512, 32, 8, 128, bf)) == 512 * 32 * 130 * 4 * 4
    for s in (sh(1, 512, 1000, 32, 8, 128, bf),     # under 512 keys a split
              sh(1, 4096, 4096, 32, 8, 128, bf),    # the grid fills the chip
              sh(1, 64, 65537, 8, 8, 128, bf),      # runs as key sub-shards
              sh(1, 512, 32512, 32, 8, 64, bf), sh(1, 512, 32512, 32, 8, 128, f32),
              sh(1, 512, 32512, 32, 8, 128, bf, _lib.LC_FLAG_PRECISE)):
        assert _bytes(lib, s) == 0
    for nq in (1, 100, 500, 2000):
        for hq in (1, 9, 32, 500):
            assert _bytes(lib, sh(1, nq, 65536, hq, 1, 128, bf)) <= 36 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("d,accumulate", [(128, False), (128, True), (64, False)])
def test_infinite_value_reaches_its_column_alone(gpu, d, accumulate):
    """An infinity in one value that every query sees: that dim of the KV head's
    rows is infinite after the merge of the splits (head_dim 64: of the waves),
    also into a running state, and the others are what they were."""
    from longctx100m_amd import ring_attention as ra

    nq, nk = 40, 3000
    rng = np.random.default_rng(d)
    q, k, v = (bf16_round(rng.standard_normal(s, dtype=np.float32))
               for s in ((1, nq, 4, d), (1, nk, 2, d), (1, nk, 2, d)))
    qt, kt, vt = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in (q, k, v))
    kw = dict(q_pos0=0, k_pos0=0, causal=False)
    eo, _, _ = dense.attention_fwd(q, k, v, **kw)
    state = {}
    if accumulate:  # the same hop before: the merge keeps o
        state = dict(zip("oml", ra.fwd_shard(qt, kt, vt, **kw)))
    vt[0, 1234, 1, 7] = float("inf")
    o, _, _ = ra.fwd_shard(qt, kt, vt, **kw, **state, accumulate=accumulate)
    got = o.cpu().numpy()
    hit = np.zeros(got.shape, bool)
    hit[0, :, 2:, 7] = True
    assert np.all(got[hit] == np.inf)
    assert norm_rel(got[~hit], eo[~hit]) <= 2e-2
