"""The ring entry points write their results from the hop kernels (no zeroing,
running copy or cast passes): the same numbers as the per-hop calls with those
passes, for every head_dim path, hops that contribute nothing, rows and keys
that no hop reaches, and results that lie over an input (written last)."""

import numpy as np
import pytest

from tests.conftest import norm_rel

pytestmark = pytest.mark.gpu

CASES = [
    # world, rank, b, n, hq, hkv, d, dtype, causal, valid
    (1, 0, 1, 1, 1, 1, 128, "bfloat16", True, None),
    (1, 0, 2, 300, 4, 2, 128, "bfloat16", True, 130),    # keys past valid_length: dk = dv = 0
    (3, 1, 1, 200, 4, 2, 128, "bfloat16", True, None),   # both passes, shared diagonal
    (3, 2, 1, 129, 4, 4, 128, "bfloat16", True, 200),    # the rank's keys invalid: zeros
    (2, 0, 1, 150, 2, 1, 64, "bfloat16", False, 150),
    (3, 1, 2, 97, 6, 2, 64, "bfloat16", True, 250),
    (2, 1, 1, 75, 4, 2, 96, "bfloat16", True, None),
    (2, 1, 1, 100, 9, 3, 64, "float32", True, 190),
    (3, 0, 1, 33, 2, 1, 40, "float32", True, None),
]


@pytest.mark.parametrize("case", CASES)
def test_ring_results_written_by_the_hops(gpu, case):
    from longctx100m_amd import ring_attention as ra

    world, rank, b, n, hq, hkv, d, dt, causal, valid = case
    rng = np.random.default_rng(n + d)
    dtype = getattr(gpu, dt)
    t = lambda h: gpu.tensor(rng.standard_normal((b, n, h, d)),  # noqa: E731
                             dtype=gpu.float32).to(dtype).cuda()
    shards = [(t(hq), t(hkv), t(hkv)) for _ in range(world)]
    grads = [t(hq) for _ in range(world)]
    kw = dict(causal=causal, valid_length=valid)
    f32 = dict(dtype=gpu.float32, device="cuda")
    fwd = []
    for r in range(world):  # per-hop calls, the running state, then a cast
        q = shards[r][0]
        o, m, l = gpu.zeros((b, n, hq, d), **f32), gpu.full((b, hq, n), -np.inf, **f32), \
            gpu.zeros((b, hq, n), **f32)
        for hop in range(world):
            w = (r - hop) % world
            ra.fwd_shard(q, shards[w][1], shards[w][2], q_pos0=r * n, k_pos0=w * n, o=o, m=m, l=l,
                         accumulate=True, **kw)
        got = ra.ring_causal_attention_forward_with_stats(shards, r, valid_length=valid,
                                                          causal=causal)
        tol = 1e-6 if dt == "float32" else 8e-3  # one bf16 rounding of o
        assert norm_rel(got[0].float().cpu(), o.cpu()) <= tol
        assert gpu.equal(got[1].view_as(m), m) and norm_rel(got[2].cpu().view_as(l), l.cpu()) <= 1e-6
        fwd.append(got)
    outs, ms, ls = (list(x) for x in zip(*fwd))

    dq = gpu.zeros((b, n, hq, d), **f32)
    dk, dv = (gpu.zeros((b, n, hkv, d), **f32) for _ in range(2))
    stats = [ra.bwd_preprocess(outs[r], grads[r], ms[r].view(b, hq, n), ls[r].view(b, hq, n))
             for r in range(world)]
    for w in range(world):
        for q_rank, k_rank, acc in ((w, rank, dict(dk_acc=dk, dv_acc=dv)), (rank, w, dict(dq_acc=dq))):
            ra.bwd_shard(shards[q_rank][0], shards[k_rank][1], shards[k_rank][2], grads[q_rank],
                         stats[q_rank][1], stats[q_rank][0], q_pos0=q_rank * n, k_pos0=k_rank * n,
                         **acc, **kw)
    tol = 2e-6 if dt == "float32" else 8e-3  # bf16: the result's rounding, and dS shared or not
    for share in (True, False):
        got = ra.ring_causal_attention_backward(shards, rank, outs, ms, ls, grads,
                                                valid_length=valid, causal=causal, share_ds=share)
        for g, e in zip(got, (dq, dk, dv)):
            assert g.dtype == dtype
            if n > 1 and not e.any():
                assert not g.any()
            elif e.abs().max() < 1e-3:  # one visible key: rounding noise
                assert (g.float() - e).abs().max() <= 2e-2
            else:
                assert norm_rel(g.float().cpu(), e.cpu()) <= tol


def test_results_over_an_input(gpu):
    """out over q in the forward, dk over k in the backward: written after the last read."""
    from longctx100m_amd import _lib
    from longctx100m_amd import ring_attention as ra

    rng = np.random.default_rng(3)
    b, n, h, d = 1, 600, 4, 128
    t = lambda: gpu.tensor(rng.standard_normal((b, n, h, d)),  # noqa: E731
                           dtype=gpu.float32).to(gpu.bfloat16).cuda()
    q, k, v, g = t(), t(), t(), t()
    want, m, l = ra.ring_causal_attention_forward_with_stats([(q, k, v)], 0)
    grads = ra.ring_causal_attention_backward([(q, k, v)], 0, [want], [m], [l], [g])
    lib, st = _lib.load(), gpu.cuda.current_stream().cuda_stream
    desc = ra._ring_desc([(q, k, v)], 0, True, 64, 128, None, None, False)
    arr = lambda x: _lib.ptr_array([x.data_ptr()])  # noqa: E731
    ws = gpu.empty(lib.lc_ring_bwd_ds_workspace_bytes(desc), dtype=gpu.uint8, device="cuda")
    q2, k2 = q.clone(), k.clone()
    keep = [arr(x) for x in (q2, k2, v, want, m, l, g)]
    m2, l2 = m.clone(), l.clone()
    _lib.check(lib.lc_ring_fwd_with_stats(desc, *(a[0] for a in keep[:3]), q2.data_ptr(),
                                          m2.data_ptr(), l2.data_ptr(), ws.data_ptr(), ws.numel(), st))
    assert gpu.equal(q2, want) and gpu.equal(m2, m)
    q2.copy_(q)
    dq, dv = gpu.empty_like(q), gpu.empty_like(v)
    _lib.check(lib.lc_ring_bwd(desc, *(a[0] for a in keep), dq.data_ptr(), k2.data_ptr(),
                               dv.data_ptr(), ws.data_ptr(), ws.numel(), st))
    for got, e in zip((dq, k2, dv), grads):
        assert norm_rel(got.float().cpu(), e.float().cpu()) <= 8e-3
