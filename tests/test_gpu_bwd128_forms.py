"""The head_dim 128 backward in each of its forms: dK/dV with four 32-key
waves per workgroup, or two key waves x four query splits (small grids), and dQ
from stored dS in workgroups of sixteen waves (up to 128 queries, and large
grids) or four; at tile edges, with and
without a diagonal, full and partial dS workspaces, against the float64 dense
oracle (bf16 bar 2e-2 norm-relative)."""

import numpy as np
import pytest

from oracle import dense
from tests.conftest import bf16_round, norm_rel

pytestmark = pytest.mark.gpu

CASES = [
    # b, nq, nk, hq, hkv, q_pos0, k_pos0, causal, valid
    # two key waves x four splits: at most 128 workgroups of 128 keys ...
    (1, 1, 1, 1, 1, 0, 0, True, None),            # one step for four groups
    (1, 33, 65, 2, 1, 40, 0, True, None),         # two steps a head, ragged key block
    (1, 95, 64, 6, 2, 0, 0, True, 50),            # nine steps over a group of three
    (2, 160, 200, 4, 1, 0, 0, True, None),        # the diagonal inside the walk
    (1, 70, 129, 2, 2, 200, 0, True, 150),        # no diagonal, valid_length
    (1, 130, 90, 3, 3, 0, 60, True, None),        # queries before every key
    # ... 256 with long walks or most keys on the diagonal, 512 with nearly all of them there
    (1, 520, 560, 48, 48, 40, 0, True, None),     # 240 workgroups
    (1, 700, 720, 90, 30, 20, 0, True, None),     # 180; four-wave dQ past 512 workgroups
    (1, 1030, 1040, 40, 40, 10, 0, True, 1037),   # 360
    # four key waves, one walk
    (1, 140, 3000, 16, 8, 2860, 0, True, None),   # 192 workgroups, walks of a few steps
    (4, 97, 300, 64, 64, 150, 0, True, None),     # 768 workgroups, diagonal
    (3, 40, 200, 66, 22, 300, 0, True, 190),      # 132, no diagonal, group of three
    (5, 33, 70, 56, 56, 20, 0, False, None),      # non-causal, 280 heads
]


@pytest.mark.parametrize("case", CASES)
def test_bwd128_forms(gpu, case):
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, qp, kp, causal, valid = case
    rng = np.random.default_rng(nq * 17 + nk)
    q, k, v, do = (bf16_round(rng.standard_normal(s, dtype=np.float32))
                   for s in ((b, nq, hq, 128), (b, nk, hkv, 128), (b, nk, hkv, 128),
                             (b, nq, hq, 128)))
    qt, kt, vt, dt = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in (q, k, v, do))
    kw = dict(q_pos0=qp, k_pos0=kp, causal=causal, valid_length=valid)
    o, m, l = ra.fwd_shard(qt, kt, vt, **kw)
    out = o.to(gpu.bfloat16)
    on = out.float().cpu().numpy()
    delta, lse2 = ra.bwd_preprocess(out, dt, m, l)
    group = hq // hkv
    want = {}
    for hk in sorted({0, hkv // 2, hkv - 1}):
        hs, ks = slice(hk * group, (hk + 1) * group), slice(hk, hk + 1)
        want[hk] = dense.attention_bwd(q[:, :, hs], k[:, :, ks], v[:, :, ks], do[:, :, hs],
                                       out=on[:, :, hs], **kw)
    full = ra.bwd_shard_workspace_bytes(qt, kt)
    per_256 = b * hq * -(-nk // 32) * 8 * 2048  # dS of 256 query rows
    for nbytes in sorted({0, full, min(full, per_256)}):
        ws = gpu.empty(nbytes, dtype=gpu.uint8, device="cuda") if nbytes else None
        acc = [gpu.zeros(x.shape, dtype=gpu.float32, device="cuda") for x in (qt, kt, vt)]
        for _ in range(2):  # the accumulators are added to
            ra.bwd_shard(qt, kt, vt, dt, lse2, delta, dq_acc=acc[0], dk_acc=acc[1],
                         dv_acc=acc[2], workspace=ws, **kw)
        got = [x.cpu().numpy() / 2 for x in acc]
        for hk, grads in want.items():
            hs, ks = slice(hk * group, (hk + 1) * group), slice(hk, hk + 1)
            for g, e, s in zip(got, grads, (hs, ks, ks)):
                if np.abs(e).max() < 1e-3:  # one visible key: the exact gradient is rounding of out
                    assert np.abs(g[:, :, s] - e).max() <= 2e-2
                else:
                    assert norm_rel(g[:, :, s], e) <= 2e-2, (nbytes, hk)
