"""Decode attention at head dim 80 on the matrix cores, whose last step of the scores is half zeros: every way the weights' pieces are laid out (as
columns of one product or as products of their own), slices of sixteen heads, lengths around a block, poisoned rows."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_decode_valu_gpu import plan
from test_parity_gpu import inputs, run_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,Hq,Hkv,L", [(2, 3, 1, 161), (3, 10, 2, 33), (1, 6, 1, 700), (2, 16, 1, 97), (2, 40, 2, 1025), (5, 12, 3, 4097), (2, 8, 4, 2500),
                                        (70, 8, 8, 385), (4, 4, 2, 31)])
@pytest.mark.parametrize("splits", [0, 1, 5])
def test_head_dim_80(lm, hip, oracle, dtype, B, Hq, Hkv, L, splits):
    D = 80
    q, k, v = inputs(oracle, (B, Hq, D), (B, Hkv, L, D), dtype, 62000 + L)
    for lens in (None, [(L, 0, 1, 32, L - 1)[i % 5] for i in range(B)]):
        kk, vv = k.copy(), v.copy()
        if lens is not None:
            for b in range(B):
                kk[b, :, lens[b]:], vv[b, :, lens[b]:] = np.nan, np.nan
        for head_map in (0, 1):
            got = run_decode(lm, hip, q, kk, vv, dtype, lens, head_map=head_map, num_splits=splits)
            want = oracle.decode_attn(q, k, v, kv_len=None if lens is None else np.array(lens, np.int32), head_map=head_map, nthreads=16)
            if lens is not None:
                want[[b for b in range(B) if lens[b] == 0]] = 0  # (zeros here, 0 / 0 there)
            assert rel_err(got, want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("splits", [1, 3])
def test_infinite_values(lm, hip, oracle, dtype, splits):
    """An infinite value reaches its own column of its KV head only, as an infinity of its sign; it lies in LDS behind a block's last row of keys."""
    q, k, v = inputs(oracle, (2, 16, 80), (2, 2, 300, 80), dtype, 62900)
    want = oracle.decode_attn(q, k, v, nthreads=16)
    for row, sign in ((0, 1), (32, -1), (299, 1)):
        w = v.copy()
        w[0, 1, row, 71] = sign * np.inf
        got = run_decode(lm, hip, q, k, w, dtype, num_splits=splits)
        assert np.array_equal(got[0, 1::2, 71], np.full(8, sign * np.inf))
        got[0, 1::2, 71] = want[0, 1::2, 71]
        assert rel_err(got, want) <= TOL[dtype]
    w[1, 0, 7, 3] = np.nan
    got = run_decode(lm, hip, q, k, w, dtype, num_splits=splits)
    assert np.isnan(got[1, ::2, 3]).all() and np.isnan(got).sum() == 8


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,Hq,Hkv,L,form", [
    (2, 3, 1, 161, "decode_mfma_kernel"), (1, 6, 1, 700, "decode_mfma_kernel"), (70, 8, 8, 385, "decode_mfma_kernel"), (9, 48, 6, 153, "decode_mfma_kernel"),
    (2, 3, 1, 160, "decode_split_kernel"), (4, 4, 2, 31, "decode_split_kernel"), (70, 8, 8, 383, "decode_split_kernel"), (1030, 3, 1, 170, "decode_split_kernel")])
def test_which_kernel(lm, hip, dtype, B, Hq, Hkv, L, form):
    """The lines of the choice, whatever the count of splits; batches that the persistent kernel does not take stay off it."""
    for splits in (0, 3):
        assert plan(lm, dtype, B, Hq, Hkv, L, 80, splits).startswith(form)
