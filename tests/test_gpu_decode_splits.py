"""The split-KV decode at the edges of its tiles, row blocks, splits and
workgroup forms, head_dim 64 and 128, against the float64 dense oracle at the
decode bars (bf16 2e-2 norm-relative; m and l within 1e-4), and its fallback
to the blockwise kernels without a usable workspace."""

import ctypes

import numpy as np
import pytest

from longctx100m_amd import _lib
from oracle import dense
from tests.conftest import bf16_round, norm_rel

# b, nq, nk, hq, hkv, d, q_pos0 offset from the cache end, k_pos0, causal, valid
CASES = [
    (1, 1, 1, 1, 1, 64, 0, 0, True, None),              # one key
    (1, 1, 63, 3, 1, 64, 0, 0, True, None),             # a partial 64-key tile
    (2, 1, 257, 9, 3, 64, 0, 0, True, None),            # five tiles for four waves
    (4, 1, 3001, 9, 3, 64, 0, 0, True, None),           # several splits
    (1, 4, 5000, 8, 2, 64, -30, 100, True, 4000),       # 16 rows, inside the cache, valid_length
    (1, 17, 100, 1, 1, 64, 0, 0, True, None),           # 17 rows: two row halves
    (2, 8, 2049, 8, 2, 64, 0, 0, True, None),           # 32 rows, head_dim 64
    (1, 11, 900, 6, 2, 128, 0, 0, True, None),          # 33 rows: a second row block of one row
    (1, 16, 1500, 4, 1, 128, -900, 0, True, None),      # 64 rows, queries inside the cache
    (1, 8, 16001, 8, 2, 128, 0, 0, True, None),         # 32 rows over many splits
    (1, 3, 40, 4, 4, 128, -39, 7, True, None),          # rows that see few keys, splits without any
    (1, 1, 500, 32, 8, 128, 0, 0, True, None),          # four tiles for each wave, one split
    (2, 4, 1000, 8, 2, 128, -500, 0, True, 700),        # tiles without a visible key after others
    (1, 1, 300000, 2, 1, 64, 0, 0, False, None),        # a long single stream: one-wave workgroups
    (1, 20, 140000, 1, 1, 128, 0, 0, True, 139000),     # the same with 32 rows
    (33, 1, 70, 16, 16, 64, 0, 0, True, None),          # more heads than the chip holds at once
]


def _rel_check(o, m, l, eo, em, el):
    fin = np.isfinite(em)
    assert norm_rel(o, eo) <= 2e-2
    assert np.array_equal(np.isfinite(m), fin) and np.all(l[~fin] == 0)
    assert np.abs(m[fin] - em[fin]).max() <= 1e-4 * max(1.0, np.abs(em[fin]).max())
    assert norm_rel(l, el) <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_decode_split_edges(gpu, case):
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, d, qoff, kp, causal, valid = case
    rng = np.random.default_rng(nq * 7 + nk + d)
    arrs = [bf16_round(rng.standard_normal(s, dtype=np.float32))
            for s in ((b, nq, hq, d), (b, nk, hkv, d), (b, nk, hkv, d))]
    q, k, v = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in arrs)
    kw = dict(q_pos0=kp + nk - nq + qoff, k_pos0=kp, causal=causal, valid_length=valid)
    o, m, l = (gpu.full(s, float("nan"), device="cuda")
               for s in ((b, nq, hq, d), (b, hq, nq), (b, hq, nq)))
    ra.decode(q, k, v, o=o, m=m, l=l, **kw)
    eo, em, el = dense.attention_fwd(*arrs, **kw)
    _rel_check(*(t.cpu().numpy() for t in (o, m, l)), eo, em, el)

    # no workspace: refused where one was always required, the blockwise kernels elsewhere
    lib = _lib.load()
    s = _lib.Shape(b, nq, nk, hq, hkv, d, _lib.LC_DTYPE_BF16, 0)
    mk = _lib.Mask(kw["q_pos0"], kp, -1 if valid is None else valid, int(causal), 0)
    ptrs = [t.data_ptr() for t in (q, k, v, o, m, l)]
    stream = gpu.cuda.current_stream().cuda_stream
    rc = lib.lc_attn_decode(ctypes.byref(s), ctypes.byref(mk), *ptrs, None, 0, stream)
    if d == 128 and nq * hq // hkv <= 16:
        assert rc == _lib.LC_ERR_WORKSPACE
    else:
        assert rc == 0
        _rel_check(*(t.cpu().numpy() for t in (o, m, l)), eo, em, el)


def test_required_workspace_sizes_are_kept():
    """head_dim 128 with at most 16 rows: one split per wave of eight per CU, at
    least two 32-key tiles each, whatever the kernel makes of it."""
    lib = _lib.load()
    for b, nq, nk, hq, hkv in ((1, 1, 262144, 32, 8), (2, 4, 3333, 8, 2), (16, 1, 64, 16, 16)):
        s = _lib.Shape(b, nq, nk, hq, hkv, 128, _lib.LC_DTYPE_BF16, 0)
        splits = max(1, min(-(-2048 // (b * hkv)), -(-nk // 32) // 2, 4096))
        need = splits * b * nq * hq * (128 * 4 + 8)
        assert lib.lc_attn_decode_workspace_bytes(ctypes.byref(s)) == -(-need // 256) * 256


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("nk", [0, 1, 3001, 300000])
def test_empty_queries_need_no_workspace(d, nk):
    """No query rows: the size query answers 0 (there is nothing to split) and
    the calls return without work, whatever the cache."""
    lib = _lib.load()
    mk = _lib.Mask(0, 0, -1, 1, 0)
    for b, hq, hkv in ((1, 9, 3), (2, 8, 8), (1, 64, 1)):
        s = _lib.Shape(b, 0, nk, hq, hkv, d, _lib.LC_DTYPE_BF16, 0)
        assert lib.lc_attn_decode_workspace_bytes(ctypes.byref(s)) == 0
        assert lib.lc_attn_fwd_shard_workspace_bytes(ctypes.byref(s)) == 0
        ptrs = [256] * 6  # never read
        assert lib.lc_attn_decode(ctypes.byref(s), ctypes.byref(mk), *ptrs, None, 0, None) == 0
        assert lib.lc_attn_decode_static(ctypes.byref(s), ctypes.byref(mk), *ptrs, None) == 0
