"""Which kernel calls with other head sizes or binary32 run, and that every plan fits its workspace
(ellm_amd/csrc/general_plan.hpp, host code)."""
import itertools

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
