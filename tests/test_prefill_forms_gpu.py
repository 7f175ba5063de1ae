"""Flash attention at the edges of the fp32 kernel's forms and of the head dims above 128: every form is reached (the
plan says so) with remainders of its row and key tiles, grouped heads and ragged keys, against the oracle."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_fused_rope_gpu import inputs, plan, rotated_on_device, run

pytestmark = pytest.mark.gpu

NT = 16


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,form", [
    (1, 2, 1, 33, 65, 16, False, "D=32, full, key groups=4> rows=16"), (1, 3, 3, 129, 70, 40, False, "D=48, full, key groups=4> rows=16"),
    (2, 32, 8, 135, 131, 64, True, "D=64, causal, key groups=2> rows=32"), (2, 40, 8, 100, 65, 72, True, "D=80, causal, key groups=2> rows=32"),
    (3, 32, 8, 500, 17, 80, False, "D=80, full, key groups=1> rows=64"), (3, 24, 24, 260, 100, 112, False, "D=112, full, key groups=1> rows=128"),
    (8, 48, 16, 257, 33, 128, True, "D=128, causal, key groups=1> rows=128"), (1, 16, 4, 1100, 1100, 96, True, "D=96, causal, key groups=2> rows=32"), (5, 30, 10, 244, 244, 64, True, "D=64, causal, key groups=1> rows=64"),
    (2, 20, 4, 637, 29, 256, False, "D=256, full, key groups=1> rows=64"),
    (1, 4, 2, 100, 300, 144, True, "D=160, causal, key groups=2> rows=32"), (1, 2, 2, 1, 1, 192, False, "D=192, full, key groups=1> rows=64"),
])
def test_fp32_forms(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, form):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), "f32", 32000 + Sq + D)
    assert "prefill_f32_kernel<" + form in plan(lm, q, k, "f32", causal, False)
    lens = [max(1, Sk - 3 * i) for i in range(B)]
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, "f32", causal, kv_len=kv_len)
        want = oracle.flash_attn(q, k, v, causal=causal, kv_len=None if kv_len is None else np.array(lens, np.int32), nthreads=NT)
        assert rel_err(got, want) <= TOL["f32"]


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("D", [144, 192, 208, 256])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (33, 63), (64, 65), (129, 300), (300, 129)])
def test_head_dims_above_128_on_the_matrix_cores(lm, hip, oracle, dtype, D, Sq, Sk):
    q, k, v = inputs(oracle, (2, 6, Sq, D), (2, 2, Sk, D), dtype, 32500 + Sq + D)
    lens = np.array([Sk, (Sk + 1) // 2], np.int32)
    for causal in (False, True):
        assert "prefill_valu_kernel" not in plan(lm, q, k, dtype, causal, False)
        got = run(lm, hip, q, k, v, dtype, causal, kv_len=lens)
        assert rel_err(got, oracle.flash_attn(q, k, v, causal=causal, kv_len=lens, nthreads=NT)) <= TOL[dtype]


def test_large_launch_of_wide_heads(lm, hip, oracle):
    # more 128-row workgroups than compute units: one key group
    q, k, v = inputs(oracle, (3, 48, 260, 256), (3, 2, 300, 256), "bf16", 32900)
    assert "key groups=1" in plan(lm, q, k, "bf16", True, False)
    assert rel_err(run(lm, hip, q, k, v, "bf16", True), oracle.flash_attn(q, k, v, causal=True, nthreads=NT)) <= TOL["bf16"]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,dtype", [
    (2, 40, 8, 385, 385, 256, True, "f16"), (3, 40, 4, 257, 330, 256, False, "bf16"), (1, 80, 8, 513, 481, 144, True, "bf16"),
    (5, 40, 8, 127, 321, 192, False, "f16"), (1, 40, 8, 1025, 1025, 208, True, "f16"), (4, 33, 3, 300, 511, 256, True, "bf16"),
])
def test_eight_waves_on_wide_heads(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, dtype):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), dtype, 32970 + Sq + D)
    assert "key groups=2, waves=8, waves per SIMD=2>" in plan(lm, q, k, dtype, causal, False)
    # a last tile with keys for both key groups, for one, and a sequence without a key (zeros; the oracle wants one)
    lens = np.array([(Sk, Sk - 30, 33, 0, 64)[i] for i in range(B)], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, dtype, causal, kv_len=None if kv_len is None else list(kv_len))
        want = oracle.flash_attn(q, k, v, causal=causal, kv_len=None if kv_len is None else np.maximum(kv_len, 1), nthreads=NT)
        if kv_len is not None:
            want[kv_len == 0] = 0
        assert rel_err(got, want) <= TOL[dtype]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,dtype,groups", [
    (2, 6, 2, 129, 129, 144, True, "bf16", 2), (5, 4, 4, 65, 321, 256, False, "f16", 2), (1, 16, 8, 700, 700, 208, True, "f16", 2),
    (2, 6, 2, 257, 500, 192, True, "bf16", 2), (3, 48, 2, 260, 300, 256, True, "bf16", 1), (4, 33, 3, 300, 190, 144, False, "f16", 1),
    (5, 32, 8, 129, 321, 192, False, "f16", 2), (1, 2, 1, 1537, 1537, 208, True, "f16", 2),  # as many key tiles in 64 rows as in 128
])
def test_a_tile_ahead_on_wide_heads(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, dtype, groups):
    """Rows of three tiles, odd ones and a last tile of one key; keys that grow along the row, so that the running maximum is
    raised again and again; sequences that end in the first tile, in its second half or before any key."""
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), dtype, 33300 + Sq + D)
    k = oracle.round_to(k * np.linspace(0.5, 8, Sk, dtype=np.float32)[:, None], dtype)
    what = plan(lm, q, k, dtype, causal, False)
    assert "key groups=%d, waves=4" % groups in what and "a tile ahead" in what
    lens = np.array([(Sk, Sk - 30, 33, 0, 64)[i] for i in range(B)], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, dtype, causal, kv_len=None if kv_len is None else list(kv_len))
        want = oracle.flash_attn(q, k, v, causal=causal, kv_len=None if kv_len is None else np.maximum(kv_len, 1), nthreads=NT)
        if kv_len is not None:
            want[kv_len == 0] = 0
        assert rel_err(got, want) <= TOL[dtype]


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("dtype,D", [("f16", 192), ("bf16", 256), ("f32", 192), ("f32", 256), ("f32", 64)])
def test_wide_heads_rotate_their_queries_in_registers(lm, hip, oracle, dtype, D, interleaved):
    q, k, v = inputs(oracle, (1, 4, 90, D), (1, 2, 90, D), dtype, 32950 + D)
    assert plan(lm, q, k, dtype, True, True) == plan(lm, q, k, dtype, True, False)
    got = run(lm, hip, q, k, v, dtype, True, rope=(7, interleaved))
    q_rot = rotated_on_device(lm, hip, q, dtype, prev_seq=7, interleaved=interleaved)
    np.testing.assert_array_equal(got, run(lm, hip, q_rot, k, v, dtype, True))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,dtype,kernel", [
    (1, 1, 1, 1000, 1000, 64, True, "f16", "key groups=2"), (1, 11, 11, 4096, 4096, 64, True, "f16", "prefill_mfma_kernel"),
    (1, 42, 42, 3000, 3000, 96, True, "f16", "prefill_mfma_pair_kernel"), (1, 50, 50, 448, 704, 64, False, "bf16", "prefill_mfma_wide_kernel"),
    (3, 7, 7, 700, 700, 128, True, "bf16", "prefill_mfma_kernel"), (1, 15, 5, 900, 900, 64, True, "f32", "prefill_f32_kernel"),
])
def test_head_counts_that_are_no_multiple_of_the_xcds(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, dtype, kernel):
    """The tiles of the heads beyond a multiple of eight go round the XCDs: every tile of every head is computed, also in
    launches that deal every other round backwards."""
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), dtype, 33000 + Sq + Hq)
    assert kernel in plan(lm, q, k, dtype, causal, False)
    assert rel_err(run(lm, hip, q, k, v, dtype, causal), oracle.flash_attn(q, k, v, causal=causal, nthreads=NT)) <= TOL[dtype]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,form", [
    (1, 32, 8, 1000, 40, 64, "D=64, key groups=1> rows=128"), (2, 15, 15, 970, 65, 56, "D=64, key groups=1> rows=128"),
    (4, 16, 4, 500, 33, 96, "D=96, key groups=1> rows=128"), (1, 31, 1, 1024, 65, 88, "D=96, key groups=1> rows=128"),
    (8, 32, 32, 127, 64, 128, "D=128, key groups=1> rows=128"), (3, 10, 5, 1001, 95, 120, "D=128, key groups=1> rows=128"),
    (3, 7, 7, 640, 320, 128, "D=128, key groups=2> rows=64"),
])
def test_fp32_without_a_mask_in_blocks_of_32(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, form):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), "f32", 33500 + Sq + D)
    assert "prefill_f32_full_kernel<" + form in plan(lm, q, k, "f32", False, False)
    # a last tile with keys for both key groups, for one, and a sequence without a key (zeros; the oracle wants one)
    lens = np.array([(Sk - 30, 0, 32, Sk)[i % 4] for i in range(B)] if B > 1 else [(Sk + 1) // 2], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, "f32", False, kv_len=None if kv_len is None else list(kv_len))
        want = oracle.flash_attn(q, k, v, kv_len=None if kv_len is None else np.maximum(kv_len, 1), nthreads=NT)
        if kv_len is not None:
            want[kv_len == 0] = 0
        assert rel_err(got, want) <= TOL["f32"]


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("Hq,Sk,D", [(32, 64, 64), (32, 64, 96), (16, 320, 128)])
def test_blocks_of_32_rotate_their_queries_in_registers(lm, hip, oracle, Hq, Sk, D, interleaved):
    q, k, v = inputs(oracle, (1, Hq, 1000, D), (1, Hq, Sk, D), "f32", 33600 + D)
    assert "prefill_f32_full_kernel" in plan(lm, q, k, "f32", False, True)
    got = run(lm, hip, q, k, v, "f32", False, rope=(7, interleaved))
    q_rot = rotated_on_device(lm, hip, q, "f32", prev_seq=7, interleaved=interleaved)
    np.testing.assert_array_equal(got, run(lm, hip, q_rot, k, v, "f32", False))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,dtype,form", [
    (13, 6, 6, 730, 730, 64, False, "f16", "key groups=1, waves=8, waves per SIMD=2>"), (10, 20, 20, 408, 65, 80, False, "f16", "key groups=1, waves=8, waves per SIMD=4>"),
    (1, 19, 19, 3000, 100, 120, False, "f16", "key groups=1, waves=4, waves per SIMD=2>"), (2, 16, 4, 777, 777, 128, True, "f16", "key groups=2, waves=4"),
    (4, 33, 11, 777, 777, 128, True, "f16", "key groups=1, waves=4, waves per SIMD=2> workgroups=928"),
    (4, 32, 8, 777, 777, 128, True, "f16", "key groups=1, waves=8, waves per SIMD=2> workgroups=448, two heads each"), (5, 20, 20, 115, 67, 64, False, "f16", "key groups=2, waves=4"),
    (5, 16, 16, 119, 119, 80, True, "bf16", "key groups=2, waves=4"), (6, 16, 4, 431, 431, 72, True, "bf16", "key groups=2, waves=4"),
    (3, 33, 11, 1285, 1285, 128, True, "bf16", "waves=4, waves per SIMD=2> workgroups=1096, V as fp16"),
])
def test_forms_chosen_by_cost(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, dtype, form):
    """Launches whose estimated cost takes them to another form than their size alone."""
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), dtype, 35000 + Sq + D)
    assert form in plan(lm, q, k, dtype, causal, False)
    lens = np.array([max(1, Sk - 31 * i) for i in range(B)], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, dtype, causal, kv_len=None if kv_len is None else list(kv_len))
        assert rel_err(got, oracle.flash_attn(q, k, v, causal=causal, kv_len=kv_len, nthreads=NT)) <= TOL[dtype]


PIECES = [(2, 16, 16, 300, 1000, 64, False, "D=64, full, key groups=2> rows=64"), (7, 24, 8, 1025, 330, 56, False, "D=64, full, key groups=2> rows=128"),
          (3, 16, 4, 700, 500, 72, False, "D=80, full, key groups=1> rows=256"), (2, 33, 3, 513, 500, 96, False, "D=96, full, key groups=1> rows=256"),
          (2, 12, 4, 1023, 401, 80, False, "D=80, full, key groups=2> rows=128"), (2, 20, 20, 300, 700, 88, False, "D=96, full, key groups=2> rows=64"),
          (2, 33, 11, 1000, 1000, 80, True, "D=80, causal, key groups=2> rows=64"), (1, 32, 8, 1300, 1300, 96, True, "D=96, causal, key groups=2> rows=128"),
          (5, 33, 33, 900, 900, 64, True, "D=64, causal, key groups=1> rows=256"), (1, 48, 4, 1100, 1100, 64, True, "D=64, causal, key groups=2> rows=64"),
          (2, 8, 2, 1000, 320, 64, False, "D=64, full, key groups=2> rows=64"), (1, 16, 8, 993, 319, 96, False, "D=96, full, key groups=2> rows=64"),
          (1, 31, 1, 1024, 97, 88, False, "D=96, full, key groups=2> rows=128")]


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,form", PIECES)
def test_fp32_on_pieces(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal, form):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), "f32", 36000 + Sq + D)
    assert "prefill_f32_split_kernel<" + form in plan(lm, q, k, "f32", causal, False)
    lens = np.array([(Sk - 30, 0, 33, Sk)[i % 4] for i in range(B)] if B > 1 else [Sk - 95], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, "f32", causal, kv_len=None if kv_len is None else list(kv_len))
        want = oracle.flash_attn(q, k, v, causal=causal, kv_len=None if kv_len is None else np.maximum(kv_len, 1), nthreads=NT)
        if kv_len is not None:
            want[kv_len == 0] = 0
        assert rel_err(got, want) <= TOL["f32"]


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("Hq,S,D", [(32, 1300, 96), (40, 1999, 64)])
def test_pieces_rotate_their_queries_in_registers(lm, hip, oracle, Hq, S, D, interleaved):
    q, k, v = inputs(oracle, (1, Hq, S, D), (1, Hq, S, D), "f32", 36100 + D)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", True, True)
    got = run(lm, hip, q, k, v, "f32", True, rope=(7, interleaved))
    q_rot = rotated_on_device(lm, hip, q, "f32", prev_seq=7, interleaved=interleaved)
    np.testing.assert_array_equal(got, run(lm, hip, q_rot, k, v, "f32", True))


@pytest.mark.parametrize("causal", [False, True])
def test_attention_on_values_that_pieces_do_not_hold(lm, hip, oracle, causal):
    """Infinities, NaN, values below the smallest normal piece and next to the largest: what fp32 gives, in the rows that see them."""
    q, k, v = inputs(oracle, (1, 40, 1000, 80), (1, 8, 1000, 80), "f32", 36200)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", causal, False)
    v[0, 0, 50, 3], v[0, 1, 60, 4] = np.inf, np.nan
    k[0, 2, 70, 5], q[0, 2::8, :, 5] = 3.4e38, q[0, 2::8, :, 5] * np.float32(2.0 ** -126)
    v[0, 3] *= np.float32(2.0 ** -122)
    k[0, 4], q[0, 4::8] = k[0, 4] * np.float32(2.0 ** -110), q[0, 4::8] * np.float32(2.0 ** 110)
    got = run(lm, hip, q, k, v, "f32", causal)
    want = oracle.flash_attn(q, k, v, causal=causal, nthreads=NT)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    for h in range(8):  # the heads of a KV head are of one magnitude
        ok = finite[0, h::8]
        err = np.abs(np.where(ok, got[0, h::8] - np.where(ok, want[0, h::8], 0), 0))
        assert err.max() <= TOL["f32"] * np.abs(want[0, h::8][ok]).max()


@pytest.mark.parametrize("Sq,D", [(1000, 80), (1999, 64), (1300, 96)])
def test_a_result_left_to_a_small_value_on_pieces(lm, hip, oracle, Sq, D):
    """The first row of a causal launch sees one key: its result is that key's value with all its bits, however far below the other
    values it lies. Keys and queries as small, beside large ones, change no weight."""
    q, k, v = inputs(oracle, (1, 40, Sq, D), (1, 8, Sq, D), "f32", 36300)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", True, False)
    for d, e in enumerate((100, 104, 108, 112, 116, 120, 124)):
        v[0, :, 0, d] *= np.float32(2.0 ** -e)
        k[0, :, 5 + d::11, d] *= np.float32(2.0 ** -e)
        q[0, ::3, d::13, d] *= np.float32(2.0 ** -e)
    got = run(lm, hip, q, k, v, "f32", True)
    for h in range(40):
        assert (np.abs(got[0, h, 0] - v[0, h % 8, 0]) <= 2.0 ** -22 * np.abs(v[0, h % 8, 0])).all()
    assert rel_err(got, oracle.flash_attn(q, k, v, causal=True, nthreads=NT)) <= TOL["f32"]


@pytest.mark.parametrize("Sq,D", [(1000, 80), (1999, 64), (1300, 96)])
def test_a_result_left_to_small_weights_on_pieces(lm, hip, oracle, Sq, D):
    """One key far ahead of all others whose value is zero: the result is the others', with weights of about 2^-121."""
    q, k, v = (np.zeros((1, n, Sq, D), np.float32) for n in (40, 8, 8))
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    q[..., 0], q[..., 1] = 1, oracle.gen_normal((1, 40, Sq), 36400)
    k[0, :, 0, 0], k[0, :, 1:, 1] = 84 * np.sqrt(D), oracle.gen_normal((8, Sq - 1), 36401)
    v[:, :, 1:] = oracle.gen_normal((1, 8, Sq - 1, D), 36402)
    got = run(lm, hip, q, k, v, "f32", False)
    s = (k[0].astype(np.float64) @ np.swapaxes(q[0, :8].astype(np.float64), 1, 2)).swapaxes(1, 2) * np.float64(np.float32(lm.default_scale(D)))
    w = np.exp(s - s.max(-1, keepdims=True))
    want = (w / w.sum(-1, keepdims=True)) @ v[0].astype(np.float64)
    # an exponent of 121 comes with an error of 2^-18 relative to one of them
    assert np.linalg.norm(got[0, :8] - want) <= 2.0 ** -17 * np.linalg.norm(want)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
def test_launches_with_very_many_heads(lm, hip, oracle, dtype):
    """More heads than a 32-bit reciprocal divides exactly: every one of them is computed."""
    B, H, Sk, D = 16384, 32, 2, 8
    q, k, v = inputs(oracle, (B, H, 1, D), (B, H, Sk, D), dtype, 34000)
    w = np.exp((q.astype(np.float64) * k).sum(-1, keepdims=True) * lm.default_scale(D))
    want = (w * v).sum(2, keepdims=True) / w.sum(2, keepdims=True)
    assert rel_err(run(lm, hip, q, k, v, dtype, False), want) <= TOL[dtype]
