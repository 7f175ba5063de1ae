"""The distribution of a flash attention launch's tiles over its workgroups, compiled for the host."""
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("deal") / "deal_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", os.path.join(HERE, "c_host", "deal_check.cpp"), "-o", binary], check=True)

    def run(lines):
        res = subprocess.run([binary], input="\n".join(lines) + "\n", stdout=subprocess.PIPE, text=True, check=True, timeout=100)
        answers = res.stdout.splitlines()
        assert len(answers) == len(lines)
        return [a for a in answers if a != "ok"]

    return run


def test_launches_with_very_many_heads(check):
    # more heads x tiles than 2^31 / heads, where a quotient through a 32-bit reciprocal is off by one
    assert not check(["%d %d %d 0 256" % s for s in [(16384, 32, 1), (4096, 64, 3), (4096, 64, 4), (2048, 64, 10), (1024, 64, 34),
                                                     (65536, 40, 1), (30011, 37, 2), (1, 524288, 3), (7, 1, 500000)]])


def test_launches_of_every_kind(check):
    rng = random.Random(7)
    shapes = [(B, Hq, tiles, res, cus) for B in (1, 2, 3) for Hq in (1, 3, 4, 8, 12, 32, 33) for tiles in (1, 2, 7, 32, 33) for res in (0, 1, 3)
              for cus in (256, 64)]
    shapes += [(rng.randint(1, 40), rng.randint(1, 70), rng.randint(1, 90), rng.randint(0, 6), rng.choice([256, 304, 38, 8])) for _ in range(300)]
    assert not check(["%d %d %d %d %d" % s for s in shapes])


def test_quotients_are_exact_for_every_31_bit_dividend(check):
    rng = random.Random(8)
    divisors = [1, 2, 3, 5, 7, 641, 65535, 65536, 65537, 2 ** 30 - 1, 2 ** 30, 2 ** 30 + 1, 2 ** 31 - 1]
    divisors += [rng.randrange(1, 1 << rng.randint(1, 31)) for _ in range(200)]
    assert not check(["divide %d" % d for d in divisors])


def test_a_launch_with_too_many_workgroups_is_refused(lm):
    p = lm.binding.AttnParams()
    p.out = p.q = p.k = p.v = 4096  # never dereferenced: the plan query stops in front of the launch
    p.B, p.Hq, p.Hkv, p.Sq, p.Sk, p.D, p.scale = 1 << 24, 64, 1, 1, 1, 64, 1.0
    for dtype in lm.binding.DTYPE_CODES.values():
        p.dtype = dtype
        with pytest.raises(lm.LuminalHipError, match="more than a launch can number"):
            lm.binding.flash_attn_plan(p)
