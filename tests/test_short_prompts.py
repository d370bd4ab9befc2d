"""Short prompts and short chunks on short caches: the kernel whose waves share a row block's keys
(short_prompt_kernel) at the edges of its tiles, and the rule that sends calls to it."""
import numpy as np
import pytest

import oracle_lib as orc
import plan_probe

# (batch, q heads, kv heads, position_index, interval, row blocks per workgroup on 256 compute units)
CASES = [
    (1, 8, 8, 0, 64, 1),         # one workgroup per 32 tokens, two key chunks for four waves
    (1, 2, 1, 0, 33, 1),         # 66 rows: two row blocks and two rows of a third
    (1, 3, 1, 95, 11, 1),        # 33 rows of a group of three, on a cache: one row in the second block
    (2, 8, 2, 0, 129, 1),        # several tokens per row block, a chunk of one key at the end
    (9, 8, 4, 7, 31, 1),         # 36 planes: one XCD each, the last four XCDs idle in the last round
    (3, 6, 1, 500, 65, 1),       # three planes: dealt round
    (1, 32, 4, 0, 1001, 2),      # two row blocks a workgroup, planes shared by two XCDs, 8 rows in the last
    (1, 64, 8, 0, 500, 2),       # 500 x 8 rows: the last workgroup holds 32 rows of 64
    (2, 48, 16, 100, 201, 2),    # 603 rows of a group of three: the last workgroup holds 27
    # few rows on a cache, calls that would stream otherwise
    (4, 32, 4, 700, 13, 1),
    (21, 32, 4, 1210, 40, 2),    # 84 planes, one XCD each
]


def test_the_rule_sends_these_calls_there():
    for b, hq, hkv, p0, s, wr in CASES:
        assert plan_probe.chunk_plan(b + 1, b, hq, hkv, p0, s)[:3] == ("short", wr, 1), (b, hq, hkv, p0, s)
    assert plan_probe.chunk_plan(1, 1, 32, 4, 0, 4096)[0] == "pingpong"       # long walks: the other kernels
    assert plan_probe.chunk_plan(1, 1, 32, 4, 8192, 64)[0] == "pingpong"
    assert plan_probe.chunk_plan(24, 24, 32, 4, 8191, 13)[:2] == ("stream", 4)


def test_calls_that_are_shorter_elsewhere_stay_there():
    """More K and V than the L2s hold, and split walks beyond 1536 keys (measured: 70.6 against 66.5 us, 53.6 against 50.3,
    38.2 against 34.4); the short-prompt kernel's own neighbours of these calls."""
    assert plan_probe.chunk_plan(6, 6, 32, 32, 1750, 150)[0] == "stream"
    assert plan_probe.chunk_plan(22, 22, 64, 8, 1329, 19)[0] == "stream"
    assert plan_probe.chunk_plan(2, 2, 32, 4, 1500, 300)[0] == "pingpong"
    assert plan_probe.chunk_plan(4, 4, 32, 32, 1600, 100)[0] == "short"      # 31 against 43 us
    assert plan_probe.chunk_plan(12, 12, 64, 8, 1506, 37)[0] == "short"      # 41 against 56
    assert plan_probe.chunk_plan(1, 1, 32, 4, 1600, 300)[0] == "short"       # 26 against 29


@pytest.mark.gpu
@pytest.mark.parametrize("flip", [False, True], ids=["", "other_type"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}x{c[4]}on{c[3]}_{c[1]}q{c[2]}kv" for c in CASES])
def test_short_prompts_match_the_oracle(case, flip):
    from gpu_util import D, LSE_TOL, compare, gpu_attention, rand_storage

    b, hq, hkv, p0, s, wr = case
    print("case", case, flush=True)
    dtype = orc.BF16 if (wr == 2) != flip else orc.F16
    q = rand_storage((s, b + 1, hq, D), 61, dtype)      # one sequence of capacity more than the batch
    k = rand_storage((b + 1, hkv, p0 + s + 1, D), 62, dtype)
    v = rand_storage((b + 1, hkv, p0 + s + 1, D), 63, dtype)
    want, want_lse = orc.attention(q, k, v, D ** -0.5, dtype, position_index=p0, batch=b)
    got, lse = gpu_attention(q, k, v, D ** -0.5, dtype, position_index=p0, batch=b)
    res = compare(got[:, :b], orc.from_storage(want, dtype)[:, :b], dtype)
    assert res["ok"], res
    assert np.abs(lse[:, :b] - want_lse[:, :b]).max() <= LSE_TOL
    assert np.isnan(got[:, b:]).all()
