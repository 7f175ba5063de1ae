"""Causal launches whose workgroups take two query heads of one KV head: both head maps, groups of two to eight heads,
ragged row tiles and lengths, head dims below the tiling, against softmax in 64 bits."""
import numpy as np
import pytest

from conftest import TOL, rel_err

pytestmark = pytest.mark.gpu


def attend(lm, hip, q, k, v, dtype, head_map, kv_len):
    args = [lm.to_device(x, hip, dtype) for x in (q, k, v)] + ([] if kv_len is None else [lm.to_device(kv_len, hip)])
    op = lm.FlashAttentionOp(lm.default_scale(q.shape[-1]), True, head_map, "f32", has_kv_len=kv_len is not None)
    return lm.execute_op(op, *args).to_host()


@pytest.mark.parametrize("B,Hkv,G,S,D,dtype,ragged", [(10, 2, 4, 1300, 128, "f16", False), (12, 2, 2, 2049, 128, "bf16", True),
                                                      (5, 3, 6, 1153, 104, "bf16", False), (9, 4, 4, 769, 112, "f16", True),
                                                      (13, 4, 2, 1030, 128, "bf16", False), (13, 2, 8, 513, 120, "f16", False),
                                                      (16, 4, 2, 1024, 128, "bf16", True), (7, 4, 2, 1994, 64, "bf16", False), (10, 4, 4, 1024, 64, "bf16", True),
                                                      (15, 3, 8, 434, 96, "f16", False), (8, 5, 4, 1792, 96, "bf16", False), (5, 3, 8, 2310, 80, "bf16", True)])
def test_two_heads_of_a_workgroup(lm, hip, oracle, B, Hkv, G, S, D, dtype, ragged):
    H = Hkv * G
    q, k, v = (oracle.round_to(oracle.gen_normal((B, h, S, D), 51000 + S + i), dtype) for i, h in enumerate((H, Hkv, Hkv)))
    lens = np.random.default_rng(S).integers(1, S + 1, size=B).astype(np.int32) if ragged else None
    if ragged:
        lens[0], lens[1] = S, 0
    rows = [0, 1, 31, 32, 127, 128, 129, S // 2, S - 130, S - 1]
    for head_map in (0, 1):
        plan = lm.flash_attention_plan(q.shape, k.shape, dtype, True)
        assert "waves=8" in plan and "two heads each" in plan
        got = attend(lm, hip, q, k, v, dtype, head_map, lens)
        for b in (0, 1, B - 1):
            n = S if lens is None else int(lens[b])
            if n == 0:
                assert not got[b].any()
                continue
            for h in range(H):
                kvh = h // G if head_map else h % Hkv
                s = q[b, h, rows].astype(np.float64) @ k[b, kvh].astype(np.float64).T / np.sqrt(D)
                s[np.arange(S)[None, :] > np.array(rows)[:, None]] = -np.inf
                s[:, n:] = -np.inf
                w = np.exp(s - s.max(1, keepdims=True))
                want = (w / w.sum(1, keepdims=True)) @ v[b, kvh].astype(np.float64)
                assert rel_err(got[b, h, rows], want) <= TOL[dtype], (b, h, head_map)
