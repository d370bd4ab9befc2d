"""How projections share K between workgroups (ellm_amd/csrc/project_plan.hpp), on the CPU: every plan is one round of
workgroups, its pieces hold at least four chunks, a handle without memory for shared sums is made without, and one with has room for the sums of every call it may run, whatever
its most rows, and for no more."""
import pytest

import plan_probe

MATRICES = ((16, 4096), (40, 2048), (96, 4096), (32, 4096), (80, 8192), (64, 8192), (1, 1024), (3, 64 * 33), (24, 5120), (85, 65536),
            (256, 8192))


def test_plans_are_well_formed():
    shared = 0
    for heads, k in MATRICES:
        for rows in (65, 79, 128, 129, 200, 256, 257, 385, 512, 640, 900, 1300):
            blocks, pieces, floats, halves = plan_probe.project_split(rows, heads, k)
            if pieces == 1:
                continue
            shared += 1
            assert pieces >= 3 and -(-rows // (128 * blocks)) * heads * pieces <= 256 and pieces * 4 <= k // 64
            assert not halves or blocks == 1
            assert floats == pieces * rows * heads * 128
    assert shared > 30


@pytest.mark.parametrize("units", [256, 200, 304])
def test_a_handle_has_room_for_every_call(units):
    shared = 0
    for heads, k in MATRICES:
        for room, need in plan_probe.project_room(heads, k, 60, 1100, units):
            assert room == need <= units * 256 * 128
            shared += need > 0
    assert shared > 4000


def test_few_rows_keep_k_whole():
    """Below 65 rows (hidden sizes the few-rows kernel does not take), whatever the handle's room."""
    for heads, k in ((1, 960), (16, 960), (40, 896)):
        assert all(plan_probe.project_split(rows, heads, k)[1] == 1 for rows in (1, 33, 64))


@pytest.mark.parametrize("status", [2, 1, 999])   # out of memory, and any other reason
def test_a_handle_without_memory_for_shared_sums(status):
    assert plan_probe.project_block(1000, 5000, 24000, status) == ([24000], 5000, 0)
    assert plan_probe.project_block(1000, 5000, 23999, status) == ([24000, 4000], 0, 0)      # K stays whole
    assert plan_probe.project_block(1000, 5000, 3999, status) == ([24000, 4000], 0, status)  # no handle
    assert plan_probe.project_block(1000, 0, 3999, status) == ([4000], 0, status)
