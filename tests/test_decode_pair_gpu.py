"""Short walks of decode attention and of decode steps, one workgroup per (sequence, KV head) pair: lengths at the edges of a wave's
32 keys and of a round of all waves (128 to 512 keys), caches whose rows past the length are NaN, every head dim and the group sizes
at which the pieces of the weights stop being columns of one product; which launches take it. Against the oracle, and steps against append + attend."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_decode_step_gpu import expected, run_step, step_inputs
from test_parity_gpu import run_decode

pytestmark = pytest.mark.gpu

CASES = [  # D, Lmax, group, dtype
    (64, 1100, 1, "f16"), (64, 513, 5, "bf16"), (64, 40, 9, "f16"), (96, 700, 4, "bf16"), (96, 385, 8, "f16"), (96, 130, 17, "bf16"),
    (128, 260, 4, "bf16"), (128, 700, 6, "bf16"), (128, 512, 8, "f16"), (128, 33, 20, "f16"), (256, 350, 2, "f16"), (256, 129, 7, "bf16"),
    (64, 1560, 3, "f16"), (96, 1040, 2, "bf16"), (128, 976, 4, "f16"), (256, 488, 1, "bf16"),
    (64, 1406, 2, "bf16"), (96, 958, 3, "f16"), (128, 859, 5, "f16"), (256, 410, 3, "bf16"),  # the longest walks of few pairs in one launch, decodes
    (64, 1562, 2, "f16"), (96, 1041, 3, "bf16"), (128, 937, 5, "bf16"), (256, 546, 3, "f16"),  # ... and steps
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


def test_steps_over_windows_of_one_buffer(lm, hip, oracle):
    """Sequences whose caches overlap attend the rows as they were before the step: a row that one of them writes may be another one's
    old row, so all are read before the first is written. Each writes another row of the buffer here."""
    B, Hq, Lmax, D, dtype = 6, 4, 96, 128, "f16"
    buf_k, buf_v = (oracle.round_to(oracle.gen_normal((Lmax + 8 * B, D), 45000 + i), dtype) for i in range(2))
    q, kn, vn = (oracle.round_to(oracle.gen_normal((B, h, D), 45010 + h + i), dtype) for i, h in enumerate((Hq, 1, 1)))
    pos = np.array([80, 61, 48, 31, 22, 5], np.int32)  # rows 80, 69, 64, 55, 54 and 45 of the buffer
    at = 8 * np.arange(B) + pos
    assert len(set(at)) == B
    dk, dv, dq, dkn, dvn = (lm.to_device(x, hip, dtype) for x in (buf_k, buf_v, q, kn, vn))
    out, dpos = lm.HipArray((B, Hq, D), "f32", hip), lm.to_device(pos, hip)
    b = lm.binding
    p, x = b.DecodeParams(), b.DecodeStepExtra()
    p.out, p.q, p.k_cache, p.v_cache, p.kv_len = out.ptr, dq.ptr, dk.ptr, dv.ptr, dpos.ptr
    p.B, p.Hq, p.Hkv, p.Lmax, p.D = B, Hq, 1, Lmax, D
    for s in (p.k_stride, p.v_stride):
        s[0], s[1], s[2] = 8 * D, D, D
    p.dtype, p.scale, p.out_f32 = b.DTYPE_CODES[dtype], lm.default_scale(D), 1
    x.k_new, x.v_new = dkn.ptr, dvn.ptr
    need = b.decode_workspace_bytes(B, Hq, 1, Lmax, D, b.decode_step_splits(B, 1, Lmax))
    scratch = lm.HipArray((need // 4,), "f32", hip).fill_bytes(0xff)
    p.workspace, p.workspace_bytes = scratch.ptr, need
    b.decode_step(p, x)
    k, v = (np.stack([w[8 * i:8 * i + Lmax] for i in range(B)])[:, None] for w in (buf_k, buf_v))
    want, _, _ = expected(oracle, q[:, :, None], kn[:, :, None], vn[:, :, None], k, v, pos, dtype, False, False, 0)
    assert rel_err(out.to_host(), want) <= TOL[dtype]
    buf_k[at], buf_v[at] = kn[:, 0], vn[:, 0]
    np.testing.assert_array_equal(dk.to_host(), buf_k)
    np.testing.assert_array_equal(dv.to_host(), buf_v)
    assert not np.isnan(scratch.to_host()).all()  # two launches


def launches(lm, hip, call):
    """How many launches a decode or a step takes: one leaves the scratch for the partial results as it is."""
    scratch = lm.host._workspaces
    at = scratch.get(1 << 25, hip)[0]
    scratch.buf.fill_bytes(0xff)
    result = call()
    assert scratch.buf.ptr == at
    return result, 1 if np.isnan(scratch.buf.to_host()).all() else 2


@pytest.mark.parametrize("B,Hkv,G,L,D,dtype,step,ragged,expected_launches", [
    (50, 4, 2, 2250, 128, "bf16", False, True, 2), (33, 7, 1, 1100, 256, "f16", False, True, 2), (28, 8, 1, 4600, 64, "f16", False, True, 2),
    (50, 4, 2, 3515, 128, "bf16", False, False, 1), (32, 8, 1, 859, 128, "f16", False, True, 1), (24, 5, 2, 585, 256, "bf16", False, True, 1),
    (45, 8, 2, 1300, 128, "f16", True, True, 1), (36, 8, 1, 660, 256, "bf16", True, True, 1), (32, 8, 2, 1406, 128, "bf16", True, True, 1),
    (28, 8, 1, 1093, 256, "f16", True, True, 1), (30, 8, 1, 1562, 64, "bf16", True, True, 1), (24, 8, 1, 1041, 96, "f16", True, True, 1),
    (55, 8, 1, 1171, 256, "bf16", True, True, 1), (40, 8, 3, 781, 64, "f16", True, True, 1), (50, 8, 1, 520, 96, "bf16", True, True, 1),
    (80, 8, 1, 170, 96, "f16", True, True, 1), (100, 8, 1, 85, 96, "f16", True, True, 1)])
def test_long_walks_of_many_pairs(lm, hip, oracle, B, Hkv, G, L, D, dtype, step, ragged, expected_launches):
    """A good part of the CUs with a pair each, or several rounds of pairs, at the longest walks that still take one launch, and decodes beyond them."""
    q, kn, vn, kc, vc = step_inputs(oracle, B, Hkv * G, Hkv, L, D, dtype, 44000 + L)
    lens = np.random.default_rng(L).integers(1, L, size=B).astype(np.int32)
    lens[:3] = (L - 1, 1, 0)
    if step:
        rope = D != 96
        (got, kc_after, vc_after), n = launches(lm, hip, lambda: run_step(lm, hip, q, kn, vn, kc, vc, lens, dtype, rope, False))
        want, _, _ = expected(oracle, q, kn, vn, kc, vc, lens, dtype, rope, False, 0)
        np.testing.assert_array_equal(vc_after[0, :, L - 1], vn[0, :, 0])
        assert rel_err(got, want) <= TOL[dtype]
    else:
        kv_len = lens if ragged else None
        got, n = launches(lm, hip, lambda: run_decode(lm, hip, q[:, :, 0], kc, vc, dtype, kv_len=kv_len, out_dtype="f32"))
        some = lens > 0 if ragged else lens >= 0
        want = oracle.decode_attn(q[some][:, :, 0], kc[some], vc[some], kv_len=lens[some] if ragged else None, nthreads=16)
        assert rel_err(got[some], want) <= TOL[dtype] and not got[~some].any()
    assert n == expected_launches


@pytest.mark.parametrize("B,Hkv,G,D,step,ragged,L,longer", [  # the longest walk in one launch (None: no walk is), and one beyond it
    (1, 8, 4, 64, True, True, 1562, 1568), (2, 8, 4, 96, True, True, 1041, 1048), (1, 8, 4, 128, True, True, 937, 944), (4, 8, 2, 256, True, True, 546, 552),
    (12, 8, 4, 128, True, True, 1093, 1100), (12, 8, 2, 256, True, True, 781, 784), (32, 8, 4, 128, True, True, 1406, 1408), (32, 8, 2, 256, True, True, 1093, 1096),
    (64, 8, 4, 128, True, True, 1328, 1336), (64, 8, 2, 256, True, True, 1168, 1176), (64, 8, 4, 64, True, True, 781, 784),
    (96, 8, 1, 64, True, True, 128, 136), (96, 8, 1, 96, True, True, 170, 176), (128, 8, 1, 96, True, True, 85, 88), (128, 8, 1, 64, True, True, None, 64),
    (1024, 8, 1, 64, True, True, None, 64), (256, 8, 4, 96, True, True, None, 64),
    (1, 8, 4, 64, False, True, 1406, 1408), (2, 8, 4, 96, False, True, 958, 960), (1, 8, 4, 128, False, True, 859, 864), (1, 8, 2, 256, False, True, 410, 416),
    (12, 8, 2, 256, False, True, 585, 592), (64, 4, 4, 128, False, False, 3515, 3520), (64, 4, 4, 128, False, True, 859, 3437), (28, 8, 1, 64, False, True, 2048, 2500)])
def test_walks_of_one_launch(lm, hip, B, Hkv, G, D, step, ragged, L, longer):
    """Caches whose lengths may differ go to one workgroup a pair only as far as one long sequence does not hold the others up."""
    for n_keys, want in ((L, 1), (longer, 2)):
        if n_keys is None:
            continue
        q, kn, vn = (lm.HipArray(shape, "f16", hip).fill_bytes(0) for shape in ((B, Hkv * G, D), (B, Hkv, 1, D), (B, Hkv, 1, D)))
        kc, vc = (lm.HipArray((B, Hkv, n_keys, D), "f16", hip).fill_bytes(0) for _ in range(2))
        lens = lm.to_device(np.full(B, n_keys - 1, np.int32), hip)
        if step:
            call = lambda: lm.execute_op(lm.DecodeStepOp(lm.default_scale(D), 0, 0, "f32", None, False), q, kc, vc, kn, vn, lens)
        else:
            call = lambda: lm.execute_op(lm.DecodeAttentionOp(lm.default_scale(D), 0, 0), q, kc, vc, *([lens] if ragged else []))
        assert launches(lm, hip, call)[1] == want, n_keys
