"""Which kernel calls with other head sizes or binary32 run, and that every plan fits its workspace
(ellm_amd/csrc/general_plan.hpp, host code)."""
import itertools
import random

import plan_probe


def test_known_calls():
    plan = plan_probe.general_plan
    assert plan(64, 2, 1, 1, 32, 8, 0, 2048)[:2] == ("chunk", 1)
    assert plan(128, 4, 8, 8, 32, 4, 4095, 1)[0] == "step"
    assert plan(64, 2, 1, 1, 32, 32, 0, 16)[0] == "rows"            # one turn of keys
    assert plan(128, 4, 1, 1, 32, 32, 0, 64)[0] == "rows"           # a short binary32 prompt
    assert plan(128, 4, 1, 1, 32, 32, 0, 300)[0] == "chunk"
    assert plan(256, 4, 1, 1, 4, 4, 100, 300)[0] == "rows"          # few rows of a wide binary32 head
    assert plan(256, 2, 1, 1, 4, 4, 100, 300)[0] == "chunk"
    assert plan(64, 4, 1, 1, 8, 2, 1900, 1)[0] == "step"


def test_a_plan_depends_on_the_rows_not_on_how_the_capacity_is_named():
    for hs, es, s in itertools.product((33, 64, 256), (2, 4), (1, 40)):
        a = plan_probe.general_plan(hs, es, 4, 2, 8, 2, 500, s)
        b = plan_probe.general_plan(hs, es, 2, 2, 8, 2, 500, s)
        assert a[0] == b[0]


def test_plans_fit_the_workspace_and_are_not_held_back_by_it():
    rng = random.Random(3)
    for _ in range(300):
        hkv = rng.choice([1, 2, 4, 8])
        hs, es, hq, b = rng.choice([19, 32, 64, 80, 128]), rng.choice([2, 4]), hkv * rng.choice([1, 3, 4, 8, 16]), rng.choice([1, 2, 5, 16])
        s, p0 = rng.choice([2, 7, 40, 130, 600]), rng.choice([0, 90, 700, 5000, 60000])
        got = plan_probe.general_plan(hs, es, b, b, hq, hkv, p0, s)
        assert got[1] == 1 or got[1] * b * hq * s <= got[5], (hs, es, hq, hkv, b, s, p0, got)
        if got[0] == "chunk":
            assert got[:5] == plan_probe.general_plan(hs, es, b, b, hq, hkv, p0, s, room=1 << 20)[:5], (hs, es, hq, hkv, b, s, p0, got)
