"""fp32 flash attention of head dims 104 to 128 on pieces of 16 bits (queries and keys as two fp16 pieces): row and key tiles with remainders,
head dims that do not fill the tiling, ragged keys, rotated queries, and values that the pieces do not hold."""
import time

import numpy as np
import pytest

from conftest import TOL, rel_err
from test_fused_rope_gpu import inputs, plan, rotated_on_device, run

pytestmark = pytest.mark.gpu

NT = 16
KERNEL = "prefill_f32_split_kernel<D=128, %s, key groups=2> rows=128"


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (2, 40, 8, 385, 385, 128, True), (1, 32, 8, 1217, 1217, 112, True), (2, 64, 8, 300, 300, 128, True), (1, 24, 8, 1030, 1030, 104, True), (3, 33, 3, 500, 321, 104, False),
    (2, 32, 8, 257, 193, 120, False), (5, 12, 6, 700, 449, 128, False), (1, 31, 1, 1024, 160, 112, False), (4, 33, 3, 250, 479, 128, False),
])
def test_tiles(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), "f32", 52000 + Sq + D)
    assert KERNEL % ("causal" if causal else "full") in plan(lm, q, k, "f32", causal, False)
    # keys for both halves of the last tile, for one, one key of it, and a sequence without any (zeros; the oracle wants one)
    lens = np.array([(Sk - 30, 33, 65, 0, Sk)[i % 5] for i in range(B)], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, "f32", causal, kv_len=None if kv_len is None else list(kv_len))
        want = oracle.flash_attn(q, k, v, causal=causal, kv_len=None if kv_len is None else np.maximum(kv_len, 1), nthreads=NT)
        if kv_len is not None:
            want[kv_len == 0] = 0
        assert rel_err(got, want) <= TOL["f32"]


@pytest.mark.parametrize("Sk,D", [(1000, 128), (513, 112)])
def test_no_further_from_64_bits_than_the_fp32_product(lm, hip, oracle, Sk, D):
    """A score is off by at most D/2 roundings of fp32 to its largest product (the fp32 product adds two at a time); normal values are far
    below that. 3e-7 is between what this kernel has (1.5e-7 to 2e-7) and what the fp32 product had (3.1e-7 to 5.7e-7)."""
    q, k, v = inputs(oracle, (1, 40, Sk, D), (1, 8, Sk, D), "f32", 52100)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    got = run(lm, hip, q, k, v, "f32", False)[0, :8].astype(np.float64)
    s = q[0, :8].astype(np.float64) @ np.swapaxes(k[0].astype(np.float64), 1, 2) * np.float64(np.float32(lm.default_scale(D)))
    w = np.exp(s - s.max(-1, keepdims=True))
    want = (w / w.sum(-1, keepdims=True)) @ v[0].astype(np.float64)
    assert np.linalg.norm(got - want) <= 3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("interleaved", [False, True])
def test_queries_rotated_in_registers(lm, hip, oracle, interleaved):
    q, k, v = inputs(oracle, (1, 32, 1300, 128), (1, 32, 1300, 128), "f32", 52200)
    assert KERNEL % "causal" in plan(lm, q, k, "f32", True, True)
    got = run(lm, hip, q, k, v, "f32", True, rope=(7, interleaved))
    q_rot = rotated_on_device(lm, hip, q, "f32", prev_seq=7, interleaved=interleaved)
    np.testing.assert_array_equal(got, run(lm, hip, q_rot, k, v, "f32", True))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [128, 104])
def test_values_that_pieces_do_not_hold(lm, hip, oracle, causal, D):
    """Infinities and NaN, queries and keys beyond fp16 and far below it: what fp32 gives, in the rows that see them."""
    q, k, v = inputs(oracle, (1, 40, 700, D), (1, 8, 700, D), "f32", 52300 + D)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", causal, False)
    v[0, 0, 50, 3], v[0, 1, 60, 4] = np.inf, np.nan
    k[0, 2, 70, 5], q[0, 2::8, :, 5] = 3.4e38, q[0, 2::8, :, 5] * np.float32(2.0 ** -126)
    k[0, 4], q[0, 4::8] = k[0, 4] * np.float32(2.0 ** -110), q[0, 4::8] * np.float32(2.0 ** 110)
    k[0, 5], q[0, 5::8] = k[0, 5] * np.float32(2.0 ** 17), q[0, 5::8] * np.float32(2.0 ** -17)
    k[0, 6], q[0, 6::8] = k[0, 6] * np.float32(2.0 ** -40), q[0, 6::8] * np.float32(2.0 ** 40)
    v[0, 3] *= np.float32(2.0 ** -122)
    got = run(lm, hip, q, k, v, "f32", causal)
    want = oracle.flash_attn(q, k, v, causal=causal, nthreads=NT)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    for h in range(8):  # the heads of a KV head are of one magnitude
        ok = finite[0, h::8]
        err = np.abs(np.where(ok, got[0, h::8] - np.where(ok, want[0, h::8], 0), 0))
        assert err.max() <= TOL["f32"] * np.abs(want[0, h::8][ok]).max()


def test_large_logits(lm, hip, oracle):
    """Scores in the hundreds, where what the pieces lack counts most: the weights' error is that of the scores, fp32's own."""
    q, k, v = inputs(oracle, (1, 40, 500, 128), (1, 8, 500, 128), "f32", 52400)
    k *= 8
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    got = run(lm, hip, q, k, v, "f32", False)
    # |s| below 60 in natural units comes with 128 products of at most 2^-22 of 30 each: 1e-4 at worst, a hundredth of it in the mean
    assert rel_err(got, oracle.flash_attn(q, k, v, nthreads=NT)) <= 1e-5


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [128, 112])
def test_magnitudes_stay_on_the_pieces(lm, hip, oracle, causal, D):
    """Powers of two taken from the keys and given to the queries, and the other way, leave every bit: both are split relative to their own
    magnitude, and none of these goes to the fp32 product, whose sums are others."""
    q, k, v = inputs(oracle, (1, 40, 700, D), (1, 8, 700, D), "f32", 52500 + D)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", causal, False)
    want = run(lm, hip, q, k, v, "f32", causal)
    for by in (-27, -17, -10, 7, 12, 27):
        got = run(lm, hip, q * np.float32(2.0 ** by), k * np.float32(2.0 ** -by), v, "f32", causal)
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("q_by,k_by", [(34, 0), (10, 24), (-20, -20), (-24, 0)])
def test_scales_stay_on_the_pieces(lm, hip, oracle, q_by, k_by):
    """The same with the power of two in the scale."""
    q, k, v = inputs(oracle, (1, 40, 520, 128), (1, 8, 520, 128), "f32", 52550)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    want = run(lm, hip, q, k, v, "f32", False)
    dq, dk, dv = (lm.to_device(x, hip, "f32") for x in (q * np.float32(2.0 ** q_by), k * np.float32(2.0 ** k_by), v))
    out = lm.HipArray(q.shape, "f32", hip)
    lm.host.execute_op_inplace(out, lm.FlashAttentionOp(float(np.float32(lm.default_scale(128)) * np.float32(2.0 ** -(q_by + k_by))), False), dq, dk, dv)
    np.testing.assert_array_equal(out.to_host(), want)


@pytest.mark.parametrize("q_mul,k_mul", [(1e3, 1e-5), (1.0, 3e3), (2e3, 1.0), (300.0, 300.0)])
def test_error_at_large_and_small_magnitudes(lm, hip, oracle, q_mul, k_mul):
    """No further from 64 bits than scores that one fp32 product after the other is added to (the softmax in 64 bits), with half as much again for
    the weights' and the result's own roundings where scores are so small that those count (3e-7 as above)."""
    q, k, v = inputs(oracle, (1, 40, 600, 128), (1, 8, 600, 128), "f32", 52600)
    q, k = q * np.float32(q_mul), k * np.float32(k_mul)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    got = run(lm, hip, q, k, v, "f32", False)[0, :8].astype(np.float64)
    scale = np.float32(lm.default_scale(128))
    chain = np.zeros((8, 600, 600), np.float32)
    for d in range(128):
        chain += q[0, :8, :, d, None] * k[0, :, None, :, d]
    exact = q[0, :8].astype(np.float64) @ np.swapaxes(k[0].astype(np.float64), 1, 2)

    def attend(s):
        s = s * np.float64(scale)
        w = np.exp(s - s.max(-1, keepdims=True))
        return (w / w.sum(-1, keepdims=True)) @ v[0].astype(np.float64)
    want = attend(exact)
    size = np.linalg.norm(want)
    assert np.linalg.norm(got - want) <= max(1.5 * np.linalg.norm(attend(chain.astype(np.float64)) - want), 3e-7 * size)


@pytest.mark.parametrize("by,most", [(2.0 ** 14, 3e-7), (2.0 ** 24, 7e-7), (2.0 ** 40, 7e-7)])  # (the pieces' error, and the fp32 product's, as above)
def test_one_large_key_among_small_ones(lm, hip, oracle, by, most):
    """The queries that turn away from it weigh the others as if it were not there: where the pieces would lose bits of those, fp32 takes over."""
    q, k, v = inputs(oracle, (1, 40, 700, 128), (1, 8, 700, 128), "f32", 52700)
    k[0, :, 70] *= np.float32(by)
    assert "prefill_f32_split_kernel" in plan(lm, q, k, "f32", False, False)
    got = run(lm, hip, q, k, v, "f32", False)
    away = np.einsum("hsd,hd->hs", q[0, :8].astype(np.float64), k[0, :, 70].astype(np.float64)) < 0
    s = q[0, :8].astype(np.float64) @ np.swapaxes(k[0].astype(np.float64), 1, 2) * np.float64(np.float32(lm.default_scale(128)))
    w = np.exp(s - s.max(-1, keepdims=True))
    want = (w / w.sum(-1, keepdims=True)) @ v[0].astype(np.float64)
    assert away.sum() > 1000
    assert np.linalg.norm((got[0, :8] - want)[away]) <= most * np.linalg.norm(want[away])


def test_large_values_take_no_longer(lm, hip, oracle):
    """Rows that go to the fp32 product as well take five times as long: queries and keys in the thousands do not."""
    q, k, v = inputs(oracle, (1, 32, 1024, 128), (1, 8, 1024, 128), "f32", 52800)
    op = lm.FlashAttentionOp(lm.default_scale(128), False)

    def best(mul):
        dq, dk, dv = (lm.to_device(x, hip, "f32") for x in (q * np.float32(mul), k * np.float32(mul), v))
        out = lm.HipArray(q.shape, "f32", hip)
        times = []
        for _ in range(8):
            lm.binding.sync()
            at = time.perf_counter()
            for _ in range(5):
                lm.host.execute_op_inplace(out, op, dq, dk, dv)
            lm.binding.sync()
            times.append(time.perf_counter() - at)
        return min(times)
    usual = best(1.0)
    for mul in (100.0, 1e3, 5e3):
        assert best(mul) < 2 * usual
