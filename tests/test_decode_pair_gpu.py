"""Short walks of decode attention and of decode steps, one workgroup per (sequence, KV head) pair: lengths at the edges of a wave's
32 keys and of a round of all waves (128 to 512 keys), caches whose rows past the length are NaN, every head dim and the group sizes
at which the pieces of the weights stop being columns of one product. Against the oracle, and steps against append + attend."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_decode_step_gpu import expected, run_step, step_inputs
from test_parity_gpu import run_decode

pytestmark = pytest.mark.gpu

CASES = [  # D, Lmax, group, dtype
    (64, 1100, 1, "f16"), (64, 513, 5, "bf16"), (64, 40, 9, "f16"), (96, 700, 4, "bf16"), (96, 385, 8, "f16"), (96, 130, 17, "bf16"),
    (128, 260, 4, "bf16"), (128, 700, 6, "bf16"), (128, 512, 8, "f16"), (128, 33, 20, "f16"), (256, 350, 2, "f16"), (256, 129, 7, "bf16"),
    (64, 1560, 3, "f16"), (96, 1040, 2, "bf16"), (128, 976, 4, "f16"), (256, 488, 1, "bf16"),  # the longest walks of few pairs
]


def lengths(Lmax, top):
    return np.array(sorted({n for n in (0, 1, 31, 32, 33, 64, 127, 128, 129, 255, 256, 257, 383, 385, 511, 513, top - 1, top) if 0 <= n <= top}), np.int32)


@pytest.mark.parametrize("D,Lmax,group,dtype", CASES)
def test_short_decode(lm, hip, oracle, D, Lmax, group, dtype):
    lens = lengths(Lmax, Lmax)
    B, Hkv = len(lens), 3
    q, _, _, k, v = step_inputs(oracle, B, Hkv * group, Hkv, Lmax, D, dtype, 41000 + D + Lmax)
    kp, vp = k.copy(), v.copy()
    for b in range(B):
        kp[b, :, lens[b]:] = np.nan
        vp[b, :, lens[b]:] = np.nan
    for head_map in (0, 1):
        got = run_decode(lm, hip, q[:, :, 0], kp, vp, dtype, kv_len=lens, head_map=head_map, out_dtype="f32")
        some = lens > 0
        want = oracle.decode_attn(q[some][:, :, 0], k[some], v[some], kv_len=lens[some], head_map=head_map, nthreads=16)
        assert rel_err(got[some], want) <= TOL[dtype]
        assert not got[~some].any()  # no key: zeros
    # without lengths: every row of the caches, and results in the caches' type
    got = run_decode(lm, hip, q[:1, :, 0], k[:1], v[:1], dtype)
    want = oracle.decode_attn(q[:1, :, 0], k[:1], v[:1], nthreads=16)
    assert rel_err(got, want) <= (2.0 ** -8 if dtype == "bf16" else 0) + TOL[dtype]


@pytest.mark.parametrize("D,Lmax,group,dtype", CASES)
def test_short_step(lm, hip, oracle, D, Lmax, group, dtype):
    pos = lengths(Lmax, Lmax - 1)
    B, Hkv = len(pos), 2
    rope, interleaved = D != 96, group % 2 == 0
    q, kn, vn, kc, vc = step_inputs(oracle, B, Hkv * group, Hkv, Lmax, D, dtype, 42000 + D + Lmax)
    kp, vp = kc.copy(), vc.copy()
    for b in range(B):
        kp[b, :, pos[b]:] = np.nan
        vp[b, :, pos[b]:] = np.nan
    got, kc_after, vc_after = run_step(lm, hip, q, kn, vn, kp, vp, pos, dtype, rope, interleaved)
    want, kc_want, _ = expected(oracle, q, kn, vn, kc, vc, pos, dtype, rope, interleaved, 0)
    assert rel_err(got, want) <= TOL[dtype]
    for b in range(B):
        np.testing.assert_array_equal(vc_after[b, :, pos[b]], vn[b, :, 0])
        assert rel_err(kc_after[b, :, pos[b]], kc_want[b, :, pos[b]]) <= (8e-3 if rope else 0)
        np.testing.assert_array_equal(kc_after[b, :, :pos[b]], kc[b, :, :pos[b]])
        assert np.isnan(kc_after[b, :, pos[b] + 1:]).all() and np.isnan(vc_after[b, :, pos[b] + 1:]).all()
    # a full cache takes no row: the result is that of the rows it has
    full = np.full(B, Lmax, np.int32)
    got, kc_after, vc_after = run_step(lm, hip, q, kn, vn, kc, vc, full, dtype, False)
    assert rel_err(got, oracle.decode_attn(q[:, :, 0], kc, vc, kv_len=full, nthreads=16)) <= TOL[dtype]
    np.testing.assert_array_equal(kc_after, kc)
    np.testing.assert_array_equal(vc_after, vc)
    # the two launches of a count of splits of the caller's, to the rounding of the sums: the caches bit for bit
    one = run_step(lm, hip, q, kn, vn, kp, vp, pos, dtype, rope, interleaved)
    two = run_step(lm, hip, q, kn, vn, kp, vp, pos, dtype, rope, interleaved, num_splits=2)
    assert rel_err(one[0], two[0]) <= 2e-6
    np.testing.assert_array_equal(one[1], two[1])
    np.testing.assert_array_equal(one[2], two[2])


@pytest.mark.parametrize("D,group,dtype", [(64, 3, "f16"), (128, 4, "bf16"), (128, 16, "f16"), (256, 2, "bf16")])
def test_new_rows_off_alignment(lm, hip, oracle, D, group, dtype):
    """New rows that do not lie on 16 bytes are loaded element by element: the same bits as of rows that do."""
    pos = np.array([0, 37, 200], np.int32)
    B, Hkv = len(pos), 2
    q, kn, vn, kc, vc = step_inputs(oracle, B, Hkv * group, Hkv, 250, D, dtype, 43000 + D + group)

    def step(shift):
        dq, dkc, dvc = lm.to_device(np.ascontiguousarray(q[:, :, 0]), hip, dtype), lm.to_device(kc, hip, dtype), lm.to_device(vc, hip, dtype)
        news = []
        for x in (kn, vn):
            whole = lm.to_device(np.concatenate([np.zeros(shift, np.float32), x.reshape(-1)]), hip, dtype)
            part = whole.view(whole.shape)
            part.shape, part.nbytes, part.ptr = x.shape, 2 * x.size, whole.ptr + 2 * shift
            news.append(part)
        out = lm.execute_op(lm.DecodeStepOp(lm.default_scale(D), 0, 0, "f32", 10000.0, False), dq, dkc, dvc, *news, lm.to_device(pos, hip))[0]
        return out.to_host(), dkc.to_host(), dvc.to_host()

    for a, b in zip(step(0), step(1)):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("B,Hkv,G,L,D,dtype,step", [(50, 4, 2, 2250, 128, "bf16", False), (33, 7, 1, 1100, 256, "f16", False), (28, 8, 1, 4600, 64, "f16", False),
                                                    (45, 8, 2, 1300, 128, "f16", True), (36, 8, 1, 660, 256, "bf16", True)])
def test_long_walks_of_many_pairs(lm, hip, oracle, B, Hkv, G, L, D, dtype, step):
    """Nearly a pair per CU, or steps whose last round of pairs is part full, at the longest walks that still take one launch."""
    q, kn, vn, kc, vc = step_inputs(oracle, B, Hkv * G, Hkv, L, D, dtype, 44000 + L)
    lens = np.random.default_rng(L).integers(1, L, size=B).astype(np.int32)
    lens[:3] = (L - 1, 1, 0)
    if step:
        got, kc_after, vc_after = run_step(lm, hip, q, kn, vn, kc, vc, lens, dtype, True, False)
        want, _, _ = expected(oracle, q, kn, vn, kc, vc, lens, dtype, True, False, 0)
        np.testing.assert_array_equal(vc_after[0, :, L - 1], vn[0, :, 0])
        assert rel_err(got, want) <= TOL[dtype]
    else:
        got = run_decode(lm, hip, q[:, :, 0], kc, vc, dtype, kv_len=lens, out_dtype="f32")
        some = lens > 0
        want = oracle.decode_attn(q[some][:, :, 0], kc[some], vc[some], kv_len=lens[some], nthreads=16)
        assert rel_err(got[some], want) <= TOL[dtype] and not got[~some].any()
