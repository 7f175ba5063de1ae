"""fp16 flash attention of head dims above 128 in four key groups, whose one tile of 128 keys is fetched K and V in turn: rows and keys at
the edges of their tiles, groups without a key (short lengths, the first causal rows), head dims that do not fill the tiling."""
import numpy as np
import pytest

from conftest import TOL, rel_err
from test_fused_rope_gpu import inputs, plan, rotated_on_device, run

pytestmark = pytest.mark.gpu

FORM = "key groups=4, waves=8"


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (1, 2, 1, 1, 2305, 256, False), (2, 4, 2, 33, 2047, 160, False), (1, 3, 3, 65, 2432, 208, False), (1, 4, 1, 300, 1281, 192, False),
    (1, 2, 2, 2337, 2337, 256, True), (1, 6, 2, 1217, 1217, 176, True), (1, 2, 1, 2000, 2300, 240, True), (2, 2, 2, 1408, 1100, 144, True),
])
def test_keys_in_turn(lm, hip, oracle, B, Hq, Hkv, Sq, Sk, D, causal):
    q, k, v = inputs(oracle, (B, Hq, Sq, D), (B, Hkv, Sk, D), "f16", 53000 + Sq + D)
    assert FORM in plan(lm, q, k, "f16", causal, False)
    short = [np.full(B, n, np.int32) for n in (1, 33, 97, 129, Sk - 1)]
    for kv_len in [None] + short:  # (one key: every group but the first has none)
        for head_map in (0, 1):
            got = run(lm, hip, q, k, v, "f16", causal, kv_len=kv_len, head_map=head_map)
            want = oracle.flash_attn(q, k, v, causal=causal, kv_len=kv_len, head_map=head_map, nthreads=16)
            assert rel_err(got, want) <= TOL["f16"]
            assert rel_err(got[:, :, :32], want[:, :, :32]) <= TOL["f16"]  # (the rows that see the fewest keys, to their own scale)


@pytest.mark.parametrize("D,S", [(256, 2500), (192, 1300)])
def test_rotated_queries_and_no_keys(lm, hip, oracle, D, S):
    """The table of the rotation's angles lies where V goes next."""
    q, k, v = inputs(oracle, (2, 2, S, D), (2, 2, S, D), "f16", 53900 + D)
    assert FORM in plan(lm, q, k, "f16", True, True)
    lens = np.array([0, 700], np.int32)
    got = run(lm, hip, q, k, v, "f16", True, rope=(3, False), kv_len=lens)
    np.testing.assert_array_equal(got, run(lm, hip, rotated_on_device(lm, hip, q, "f16", prev_seq=3), k, v, "f16", True, kv_len=lens))
    assert not got[0].any()


def test_lines_of_the_choice(lm, oracle):
    """Shorter walks, bf16 and launches that fill the CUs with higher workgroups stay where they are."""
    def name(B, H, S, D, dtype="f16"):
        q, k, _ = inputs(oracle, (B, H, S, D), (B, H, 1, D), dtype, 1)
        return plan(lm, q, np.broadcast_to(k, (B, H, S, D)), dtype, True, False)
    assert FORM in name(1, 2, 2400, 256) and FORM in name(1, 2, 1200, 160)
    for call in [(1, 2, 1500, 256), (1, 2, 600, 160), (1, 2, 2400, 256, "bf16"), (4, 16, 2400, 256)]:
        assert FORM not in name(*call)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(1, 6, 7218, 7218, 256, True), (5, 4, 961, 961, 192, True), (3, 6, 1148, 1148, 192, True), (5, 32, 252, 4832, 176, False),
                                                (14, 4, 674, 6304, 208, False)])
def test_launches_of_more_workgroups_than_cus_stay(lm, B, H, Sq, Sk, D, causal):
    name = lm.flash_attention_plan((B, H, Sq, D), (B, H, Sk, D), "f16", causal)
    assert FORM not in name, name
