"""Causal launches whose row tiles do not fill their rows: the tiles begin before row 0. Lengths around multiples of the key tile and of
every row tile (64, 128, 256 and pairs of 256 rows; 16 to 128 in fp32), with short keys, with lengths per sequence and rotated queries."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_fused_rope_gpu import inputs, plan, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,dtype,form", [
    (1, 3, 1, 65, 65, 64, "f16", "key groups=2, waves=4"), (2, 5, 5, 191, 191, 80, "bf16", "key groups=2, waves=4"),
    (2, 32, 4, 1151, 1151, 128, "f16", "key groups=1, waves=4"), (6, 32, 8, 833, 833, 64, "f16", "key groups=1, waves=4"),
    (2, 32, 8, 1100, 900, 128, "bf16", "key groups=1, waves=4"), (2, 64, 8, 1153, 1153, 96, "f16", "waves=8, waves per SIMD=4"),
    (2, 32, 8, 2177, 2177, 128, "bf16", "waves=8, waves per SIMD=2> workgroups=576, two heads each, V as fp16"), (2, 32, 8, 2177, 2177, 128, "f16", "waves=8, waves per SIMD=2"),
    (4, 33, 3, 300, 511, 256, "bf16", "waves=8"), (1, 128, 16, 833, 833, 96, "f16", "pair_kernel"), (3, 85, 5, 385, 1000, 64, "f16", "pair_kernel"),
    (2, 20, 4, 577, 577, 64, "f32", "prefill_f32_split_kernel<D=64, causal, key groups=2> rows=64"),
    (1, 32, 8, 1217, 1217, 96, "f32", "prefill_f32_split_kernel<D=96, causal, key groups=2> rows=128"),
    (1, 40, 8, 65, 200, 64, "f32", "prefill_f32_kernel<D=64, causal, key groups=4> rows=16"),
    (1, 40, 8, 300, 300, 128, "f32", "prefill_f32_kernel<D=128, causal, key groups=2> rows=32"),
    (1, 64, 4, 1100, 1100, 112, "f32", "prefill_f32_kernel<D=112, causal, key groups=1> rows=128"),
])
def test_short_first_tile(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, dtype, form):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), dtype, 43000 + Sq + D)
    assert form in plan(lm, q, k, dtype, True, False)
    lens = np.array([max(1, Sk - 70 * i) for i in range(B)], np.int32)
    for kv_len in (None, lens):
        got = run(lm, hip, q, k, v, dtype, True, kv_len=kv_len)
        want = oracle.flash_attn(q, k, v, causal=True, kv_len=kv_len, nthreads=16)
        assert rel_err(got, want) <= TOL[dtype]
        assert rel_err(got[:, :, :64], want[:, :, :64]) <= TOL[dtype]  # (the rows whose tile is short, to their own scale)
