"""Decode attention on the vector ALUs (fp32, and head dims that the matrix-core kernel does not tile) where the count of splits is open: short walks
in one split, on four or sixteen waves, and a wide workgroup per CU for few long ones. Lengths around the keys of an iteration, sequences
without keys, rows past the length poisoned; and the counts of a caller, which stay."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_parity_gpu import inputs, run_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,Hq,Hkv,L,D", [
    ("f32", 3, 2, 2, 229, 64), ("f32", 2, 12, 6, 243, 128), ("f32", 4, 8, 2, 153, 256), ("f32", 5, 64, 8, 77, 96), ("f32", 1, 3, 3, 615, 64),
    ("f32", 40, 8, 8, 152, 64), ("f32", 24, 24, 12, 202, 128), ("f32", 3, 5, 5, 448, 36),
    ("f16", 3, 8, 8, 513, 80), ("bf16", 5, 4, 2, 300, 80), ("f16", 6, 16, 4, 150, 80), ("bf16", 9, 48, 6, 153, 80), ("f16", 25, 12, 12, 447, 80),
    ("bf16", 70, 24, 4, 255, 80), ("f16", 2, 7, 7, 230, 248),
    ("bf16", 1, 2, 2, 29834, 80), ("f16", 3, 4, 4, 8211, 80), ("f32", 2, 4, 2, 7376, 256), ("f32", 1, 16, 4, 9001, 128), ("f32", 6, 1, 1, 11075, 64)])
def test_open_counts(lm, hip, oracle, dtype, B, Hq, Hkv, L, D):
    q, k, v = inputs(oracle, (B, Hq, D), (B, Hkv, L, D), dtype, 61000 + L + D)
    for lens in (None, [max(0, L - 31 * i) for i in range(B)], [(1, 0, L, 33, 65, L // 2)[i % 6] for i in range(B)]):
        kk, vv = k.copy(), v.copy()
        if lens is not None:
            for b in range(B):  # rows that no sequence has
                kk[b, :, lens[b]:], vv[b, :, lens[b]:] = np.nan, np.nan
        for head_map in (0, 1):
            got = run_decode(lm, hip, q, kk, vv, dtype, lens, head_map=head_map)
            want = oracle.decode_attn(q, k, v, kv_len=None if lens is None else np.array(lens, np.int32), head_map=head_map, nthreads=16)
            if lens is not None:
                want[[b for b in range(B) if lens[b] == 0]] = 0  # (zeros here, 0 / 0 there)
            assert rel_err(got, want) <= TOL[dtype]
            # a caller's own count: the same sums in another order
            assert rel_err(run_decode(lm, hip, q, kk, vv, dtype, lens, head_map=head_map, num_splits=3), want) <= TOL[dtype]


def plan(lm, dtype, B, Hq, Hkv, L, D, num_splits=0):
    p = lm.binding.DecodeParams()
    p.out = p.q = p.k_cache = p.v_cache = p.workspace = 4096
    p.B, p.Hq, p.Hkv, p.Lmax, p.D = B, Hq, Hkv, L, D
    p.dtype, p.scale, p.num_splits, p.workspace_bytes = lm.binding.DTYPE_CODES[dtype], lm.default_scale(D), num_splits, 1 << 40
    return lm.binding.decode_plan(p)


@pytest.mark.parametrize("dtype,B,Hq,Hkv,L,D,form", [
    # one split: eight heads a workgroup, more units than CUs, and both; walks for sixteen waves; four heads
    ("bf16", 9, 48, 6, 70, 72, "lanes a key=16, heads=8, waves=4> splits=1"), ("f16", 70, 24, 4, 255, 112, "lanes a key=16, heads=8, waves=4> splits=1"),
    ("f16", 92, 12, 12, 131, 80, "lanes a key=16, heads=1, waves=4> splits=1"), ("bf16", 25, 12, 12, 447, 160, "lanes a key=32, heads=1, waves=4> splits=1"),
    ("f16", 3, 8, 8, 513, 80, "lanes a key=16, heads=1, waves=16> splits=1"), ("bf16", 5, 8, 4, 301, 72, "lanes a key=16, heads=2, waves=16> splits=1"),
    ("bf16", 6, 24, 6, 75, 160, "lanes a key=32, heads=4, waves=4> splits=1"), ("f32", 40, 8, 8, 152, 64, "lanes a key=16, heads=1, waves=4> splits=1"),
    ("f32", 2, 12, 6, 151, 256, "lanes a key=64, heads=2, waves=16> splits=1"), ("f32", 7, 36, 3, 201, 32, "lanes a key=8, heads=8, waves=4> splits=1"),
    # two heads, longer than two iterations of sixteen waves: partials
    ("f16", 2, 12, 6, 575, 72, "lanes a key=16, heads=2, waves=4> splits=5"), ("bf16", 8, 16, 8, 613, 72, "lanes a key=16, heads=2, waves=16> splits=1"),
    ("f16", 50, 2, 1, 258, 192, "lanes a key=32, heads=2, waves=16> splits=1"),
    # few units: a wide workgroup a CU
    ("f16", 1, 4, 1, 30001, 112, "lanes a key=16, heads=4, waves=8> splits="), ("bf16", 3, 3, 1, 16385, 200, "lanes a key=32, heads=4, waves=8> splits="),
    ("bf16", 1, 2, 2, 29834, 80, "lanes a key=16, heads=1, waves=16> splits="), ("f32", 6, 1, 1, 11075, 64, "lanes a key=16, heads=1, waves=16> splits="),
])
def test_forms(lm, hip, oracle, dtype, B, Hq, Hkv, L, D, form):
    """Each form of the kernel, by name: its lanes, heads and waves."""
    assert ("decode_split_kernel<%s, " % dtype + form) in plan(lm, dtype, B, Hq, Hkv, L, D)
    q, k, v = inputs(oracle, (B, Hq, D), (B, Hkv, L, D), dtype, 63000 + L + D)
    lens = [(L, max(L - 33, 1), 0, 1, L // 2 + 1)[i % 5] for i in range(B)]
    for b in range(B):  # rows that no sequence has
        k[b, :, lens[b]:], v[b, :, lens[b]:] = 0, 0
    kk, vv = k.copy(), v.copy()
    for b in range(B):
        kk[b, :, lens[b]:], vv[b, :, lens[b]:] = np.nan, np.nan
    for head_map in (0, 1):
        got = run_decode(lm, hip, q, kk, vv, dtype, lens, head_map=head_map)
        want = oracle.decode_attn(q, k, v, kv_len=np.array(lens, np.int32), head_map=head_map, nthreads=16)
        want[[b for b in range(B) if lens[b] == 0]] = 0  # (zeros here, 0 / 0 there)
        assert rel_err(got, want) <= TOL[dtype]


@pytest.mark.parametrize("dtype,D", [("f32", 64), ("f16", 80), ("bf16", 80)])
def test_infinities_stay_in_their_rows(lm, hip, oracle, dtype, D):
    """An infinite value row reaches the heads that attend it and no other, whatever the waves without a key load."""
    q, k, v = inputs(oracle, (2, 4, D), (2, 4, 300, D), dtype, 61900)
    v[0, 1, 299, 3] = np.inf
    got = run_decode(lm, hip, q, k, v, dtype, [300, 299])
    assert np.isposinf(got[0, 1, 3])
    got[0, 1, 3] = 0
    v[0, 1, 299, 3] = 0
    want = oracle.decode_attn(q, k, v, kv_len=np.array([300, 299], np.int32), nthreads=16)
    want[0, 1, 3] = 0
    assert rel_err(got, want) <= TOL[dtype]
