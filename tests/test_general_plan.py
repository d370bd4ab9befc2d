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


def test_the_form_of_the_chunk_kernel():
    """Heads of 65 to 96 with one key group: the maximum every step from three workgroups a unit (256) on, and from
    two on where what those leave is not short."""
    def every_step(*call):
        return plan_probe.general_plan(96, 2, call[0], *call)[6]

    assert not every_step(4, 32, 32, 0, 512) and not every_step(1, 32, 8, 0, 1600)      # 512, 400 workgroups
    assert every_step(4, 32, 32, 0, 700) and every_step(4, 32, 32, 0, 2048)             # 768, 2048
    assert not every_step(2, 32, 8, 0, 1400) and every_step(2, 32, 8, 500, 1300)        # 704, the last short; 656, all long
    assert not every_step(3, 32, 32, 0, 700) and every_step(7, 32, 32, 0, 300)          # 576 and 672 with few row tiles a plane
    for hs, want in ((64, 0), (128 - 8, 0), (192, 1)):
        assert plan_probe.general_plan(hs, 2, 4, 4, 32, 32, 0, 700)[6] == want


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
