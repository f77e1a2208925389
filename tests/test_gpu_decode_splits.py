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
    (1, 1, 1, 1, 1, 64, 0, 0, True, None),              # one key: the blockwise kernel, as up to
    (1, 1, 1024, 3, 1, 64, 0, 0, True, None),           # 1,024 keys of few sequences
    (1, 1, 1025, 3, 1, 64, 0, 0, True, None),           # 17 tiles, the last of one key
    (9, 1, 63, 32, 8, 64, 0, 0, True, None),            # one split: a partial 64-key tile
    (9, 1, 300, 32, 8, 64, 0, 0, True, None),           # five tiles for four waves
    (9, 8, 300, 32, 8, 64, 0, 0, True, None),           # the same with 32 rows
    (5, 8, 300, 64, 8, 64, -40, 0, True, 290),          # and with 64
    (9, 8, 70, 32, 8, 128, 0, 0, True, None),           # one split, head_dim 128, 32 rows
    (5, 8, 300, 64, 8, 128, -40, 0, True, 290),         # and 64
    (4, 1, 3001, 9, 3, 64, 0, 0, True, None),           # several splits
    (1, 4, 5000, 8, 2, 64, -30, 100, True, 4000),       # 16 rows, inside the cache, valid_length
    (1, 17, 100, 1, 1, 64, 0, 0, True, None),           # 17 rows, few keys: blockwise
    (1, 17, 1500, 1, 1, 64, 0, 0, True, None),          # 17 rows: two row halves
    (1, 16, 3000, 8, 2, 64, 0, 0, True, None),          # 64 rows: two row blocks of 32
    (1, 13, 3000, 10, 2, 64, 0, 0, True, None),         # 65: blockwise
    (1, 13, 3000, 10, 2, 128, 0, 0, True, None),        # the same, head_dim 128
    (1, 9, 2100, 8, 1, 128, -100, 0, True, None),       # 72
    (2, 8, 2049, 8, 2, 64, 0, 0, True, None),           # 32 rows, head_dim 64
    (1, 11, 900, 6, 2, 128, 0, 0, True, None),          # 33 rows: a second row block of one row
    (1, 16, 1500, 4, 1, 128, -900, 0, True, None),      # 64 rows, queries inside the cache
    (1, 8, 16001, 8, 2, 128, 0, 0, True, None),         # 32 rows over many splits
    (1, 3, 40, 4, 4, 128, -39, 7, True, None),          # rows that see few keys, splits without any
    (1, 1, 500, 32, 8, 128, 0, 0, True, None),          # four tiles for each wave, one split
    (2, 4, 1000, 8, 2, 128, -500, 0, True, 700),        # tiles without a visible key after others
    (1, 1, 300000, 2, 1, 64, 0, 0, False, None),        # a long single KV head: four waves each
    (1, 1, 140001, 6, 6, 64, 0, 0, False, None),        # a long single stream: one-wave workgroups
    (1, 5, 140001, 24, 6, 64, 0, 0, True, 139000),      # the same with 32 rows
    (1, 5, 70001, 24, 6, 128, 0, 0, True, None),        # and head_dim 128
    (33, 1, 70, 16, 16, 64, 0, 0, True, None),          # more heads than the chip holds: blockwise
]

# Splits of the shapes above that use a workspace, None where the blockwise
# kernel runs, 1 where one workgroup takes all keys.  One-wave workgroups are
# as many as the chip has wave slots, rounded up (2,048 / 6 -> 342; four-wave
# ones round down).
SPLITS = {
    (1, 1, 1024, 3, 1, 64): None, (9, 1, 300, 32, 8, 64): 1, (9, 8, 300, 32, 8, 64): 1,
    (5, 8, 300, 64, 8, 64): 1, (9, 8, 70, 32, 8, 128): 1, (5, 8, 300, 64, 8, 128): 1,
    (1, 17, 100, 1, 1, 64): None, (1, 13, 3000, 10, 2, 64): None, (1, 13, 3000, 10, 2, 128): None,
    (1, 9, 2100, 8, 1, 128): None, (33, 1, 70, 16, 16, 64): None,
    (1, 1, 1025, 3, 1, 64): 5, (1, 17, 1500, 1, 1, 64): 6, (1, 16, 3000, 8, 2, 64): 12,
    (1, 1, 140001, 6, 6, 64): 342, (1, 5, 140001, 24, 6, 64): 342, (1, 5, 70001, 24, 6, 128): 342,
}


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


@pytest.mark.parametrize("shape", SPLITS)
def test_cases_take_the_form_they_name(shape):
    """The workspace size tells the number of splits, and with it the form."""
    lib = _lib.load()
    b, nq, nk, hq, hkv, d = shape
    assert shape in [c[:6] for c in CASES]
    s = _lib.Shape(b, nq, nk, hq, hkv, d, _lib.LC_DTYPE_BF16, 0)
    need = SPLITS[shape] * b * nq * hq * (d * 4 + 8) if (SPLITS[shape] or 1) > 1 else 0
    assert lib.lc_attn_decode_workspace_bytes(ctypes.byref(s)) == -(-need // 256) * 256


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1, 4001, 8, 2, 128), (1, 5, 4001, 8, 2, 128),
                                   (1, 1, 500, 8, 2, 128), (2, 1, 4001, 6, 2, 64),
                                   (1, 1, 70001, 12, 12, 128)])
def test_infinite_value_reaches_its_column_alone(gpu, shape):
    """An infinity in one visible value makes that dim of the rows infinite,
    through the waves' and the splits' merges, and leaves the others."""
    from longctx100m_amd import ring_attention as ra

    b, nq, nk, hq, hkv, d = shape
    rng = np.random.default_rng(nk)
    arrs = [bf16_round(rng.standard_normal(s, dtype=np.float32))
            for s in ((b, nq, hq, d), (b, nk, hkv, d), (b, nk, hkv, d))]
    eo, _, _ = dense.attention_fwd(*arrs, causal=False, q_pos0=0, k_pos0=0)
    q, k, v = (gpu.tensor(x).to(gpu.bfloat16).cuda() for x in arrs)
    v[0, nk // 3, hkv - 1, 5] = float("inf")
    o, _, _ = ra.decode(q, k, v, q_pos0=0, causal=False)
    got = o.cpu().numpy()
    hit = np.zeros(got.shape, bool)
    hit[0, :, hq - hq // hkv:, 5] = True
    assert np.all(got[hit] == np.inf)
    assert norm_rel(got[~hit], eo[~hit]) <= 2e-2


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
