"""The reference maximum of the chunk kernel for other 16-bit heads: moved by score levels that pass its step once,
again and again or in some rows of a block only, with one, two and four key groups, key splits and rows that are not
whole 16-byte pieces.  Heads up to 128 look for a row's maximum only where a lane's sum of weights asks for it, wider
ones every step."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from gpu_util import LSE_TOL, storage_ulp
from test_gpu_general_heads import _run

pytestmark = pytest.mark.gpu

# levels of successive runs of 128 keys (a step or more of every key group), in units of the score's log2
LEVELS = {"below": [0, 7, 6, 7], "once": [0, 0, 17, 17], "rising": [0, 16, 40, 300], "falling": [300, 30, 10, 0],
          "waves": [0, 40, -40, 60]}

# (head size, sequences, query heads, key-value heads, position_index, interval), (key groups, splits, maximum every step)
CASES = [((64, 1, 8, 2, 450, 50), (4, 1, 0)), ((64, 1, 8, 1, 2000, 70), (4, 5, 0)), ((64, 5, 64, 64, 400, 129), (2, 1, 0)),
         ((80, 1, 4, 1, 520, 100), (4, 2, 0)), ((96, 16, 32, 8, 430, 130), (1, 1, 1)), ((80, 4, 32, 32, 0, 500), (1, 1, 0)),
         ((33, 2, 4, 2, 440, 50), (4, 1, 0)),
         ((24, 1, 4, 1, 450, 60), (4, 1, 0)), ((192, 1, 8, 2, 450, 60), (2, 1, 1))]


@pytest.mark.parametrize("case,cut", CASES, ids=["h%d_b%d_%dq%d_%d+%d" % c[0] for c in CASES])
@pytest.mark.parametrize("name", LEVELS)
@pytest.mark.parametrize("dtype", [orc.F16, orc.BF16], ids=["f16", "bf16"])
def test_scores_that_outgrow_the_reference(case, cut, name, dtype):
    hs, b, hq, hkv, p0, s = case
    print("case", case, name, flush=True)
    plan = plan_probe.general_plan(hs, 2, b, b, hq, hkv, p0, s)
    assert plan[0] == "chunk" and (plan[3], plan[1], plan[6]) == cut
    cap = p0 + s
    scale = 1.0 / math.sqrt(hs)
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal(n, dtype=np.float32) for n in ((s, b, hq, hs), (b, hkv, cap, hs), (b, hkv, cap, hs)))
    q[..., 0] = 8.0 * (np.arange(s)[:, None, None] % 3 - 1)    # of three rows one rises, one falls, one stays
    level = np.array([LEVELS[name][(i // 128) % 4] for i in range(cap)], dtype=np.float32)
    k[..., 0] = level * np.float32(math.log(2.0) / (8.0 * scale))
    q, k, v = (orc.to_storage(a, dtype) for a in (q, k, v))
    got, lse = _run(q, k, v, scale, dtype, p0=p0)
    want, want_lse = orc.attention(q, k, v, scale, dtype, position_index=p0)
    want = orc.from_storage(want, dtype)
    # A weight goes in as two storage values, to 2^-17 of it (bfloat16) or 2^-22 (binary16), and binary32 sums over 2000
    # keys in another order stay below 2^-16 of the values' weighted magnitudes.  A score of magnitude L is itself a
    # binary32 sum of up to 192 products, one of which is nearly all of it: every later addition rounds by up to
    # 2^-25 L, which moves the weight by as much of itself, sixteen times on either side if two in three cancel.
    # Both sides round the output once.
    weight = 2.0 ** -16 + 32 * 2.0 ** -25 * max(abs(x) for x in LEVELS[name]) * math.log(2.0)
    mags = orc.to_storage(np.abs(orc.from_storage(v, dtype)), dtype)
    size = orc.from_storage(orc.attention(q, k, mags, scale, dtype, position_index=p0)[0], dtype)
    err, bound = np.abs(got - want), weight * size + storage_ulp(want, dtype)
    assert (err <= bound).all(), float((err / bound).max())
    # (a log-sum-exp of up to 208 is spaced 2^-16; the bound leaves it a dozen roundings)
    assert np.abs(lse - want_lse).max() <= LSE_TOL + 12 * 2.0 ** -16
