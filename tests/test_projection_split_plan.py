"""How projections share K between workgroups (ellm_amd/csrc/project_plan.hpp), on the CPU: every plan is one round of
workgroups, its pieces hold at least four chunks, its sums fit what a handle for that many rows takes, and with less
room they fit that or K stays whole."""
import plan_probe


def test_plans_are_well_formed_and_fit():
    shared = 0
    for heads, k in ((16, 4096), (40, 2048), (96, 4096), (32, 4096), (80, 8192), (64, 8192), (1, 1024), (3, 64 * 33), (85, 65536), (256, 8192)):
        for rows in (65, 79, 128, 129, 200, 256, 257, 385, 512, 640, 900, 1300):
            blocks, pieces, floats, room, halves = plan_probe.project_split(rows, heads, k)
            if pieces == 1:
                continue
            shared += 1
            assert pieces >= 3 and -(-rows // (128 * blocks)) * heads * pieces <= 256 and pieces * 4 <= k // 64
            assert not halves or blocks == 1
            assert floats == pieces * rows * heads * 128 <= room <= 256 * 256 * 128
            tight = plan_probe.project_split(rows, heads, k, floats - 1)
            assert tight[1] == 1 or tight[2] < floats
    assert shared > 30
