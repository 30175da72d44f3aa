"""Splits of a last round of more than half the slots: over several rounds, only
where they beat an unsplit round of a partly idle chip."""

import random

import pytest

from moonmath_attention import _lib
from oracle import planner


@pytest.mark.parametrize("ctas,nkb,want", [
    # 144 CTAs: a round's blocks at 45 + 55*144/256 = 75%, so 76% of 192 + 4 = 148;
    # 3 parts: 432 CTAs, 64 * (100 + 82)% + 2*4 + 3 + 11 = 138; of 48: 40 against 51.
    (144, 48, (144, 0, 1, 0)),
    (144, 192, (0, 144, 3, 432)),
    (192, 192, (192, 0, 1, 0)),
    (456, 192, (456, 0, 1, 0)),
    (400, 192, (256, 144, 3, 432)),
    # Half the slots and fewer: one round of parts.
    (128, 192, (0, 128, 2, 256)),
    (129, 48, (129, 0, 1, 0)),
    (96, 192, (0, 96, 2, 192)),
])
def test_last_rounds(ctas, nkb, want):
    assert planner.plan_tail(ctas, 1, nkb, 256, 1024) == want
    assert _lib.plan_tail(1, 1, ctas * 256, nkb * 64) == want


def test_host_planner_is_the_oracles():
    rng = random.Random(3)
    for _ in range(2000):
        ctas, nkb = rng.randint(1, 1200), rng.randint(1, 2000)
        got = _lib.plan_tail(1, 1, ctas * 256, nkb * 64)
        assert got == planner.plan_tail(ctas, 1, nkb, 256, 1024), (ctas, nkb)
        assert got[3] <= 1024 and got[0] + got[1] == ctas
