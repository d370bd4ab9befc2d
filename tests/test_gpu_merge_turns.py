"""The merge launch of split chunk calls: counts of pieces below, at and above what a lane takes at once and what lanes
share (one lane up to eight pieces or in large grids, eight lanes to 32, 64 lanes beyond), 128-wide heads and others.
Same oracle and bounds as tests/test_gpu_random_shapes.py and tests/test_gpu_general_heads.py; values so large that the pieces'
sums only add up within binary32 under the weights of the row's final maximum, against the closed form."""
import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from gpu_util import D, LSE_TOL, compare, gpu_attention, rand_storage
from test_gpu_general_heads import _check, _rand, _run

pytestmark = pytest.mark.gpu

# pieces, batch, q heads, kv heads, position_index, interval
WIDE = [(2, 64, 8, 4, 500, 2), (3, 40, 32, 4, 1000, 2), (4, 1, 16, 1, 2000, 33), (5, 1, 16, 1, 2500, 33), (6, 1, 4, 4, 1700, 2),
        (9, 12, 4, 4, 3300, 2), (10, 1, 16, 1, 5000, 33), (10, 1, 32, 4, 4704, 70), (16, 1, 4, 4, 5000, 2),
        (20, 1, 16, 1, 5000, 9), (29, 1, 4, 4, 9000, 2), (36, 1, 16, 1, 9000, 9), (94, 1, 4, 1, 24000, 2), (240, 1, 4, 1, 76798, 2)]
# pieces, head size, batch, q heads, kv heads, position_index, interval
OTHER = [(2, 64, 1, 8, 1, 600, 5), (3, 64, 1, 8, 1, 1100, 5), (4, 64, 1, 8, 1, 1700, 5), (5, 64, 1, 8, 1, 2500, 5),
         (9, 64, 1, 8, 1, 4200, 5), (10, 256, 1, 8, 1, 2400, 140), (16, 64, 2, 4, 4, 9000, 70), (18, 64, 1, 8, 1, 9000, 5)]
GRID = (1 << 19) // 8       # (row, four columns) items beyond which one lane takes all pieces


def _ids(cases):
    return ["%d_pieces_%d" % (c[0], c[-1]) for c in cases]


def test_cases_reach_one_lane_beyond_the_small_grids():
    assert any(n > 8 and b * hq * s * 32 > GRID for n, b, hq, _, _, s in WIDE)
    assert any(n > 8 and b * hq * s * ((hs + 31) // 32 * 8) > GRID for n, hs, b, hq, _, _, s in OTHER)


@pytest.mark.parametrize("pieces,b,hq,hkv,p0,s", WIDE, ids=_ids(WIDE))
def test_pieces_of_wide_heads(pieces, b, hq, hkv, p0, s):
    print("pieces", pieces, b, hq, hkv, p0, s, flush=True)
    assert plan_probe.chunk_plan(b, b, hq, hkv, p0, s)[2] == pieces
    dtype = orc.BF16 if pieces % 2 else orc.F16
    q, k, v = (rand_storage(n, 610 + i, dtype) for i, n in enumerate(((s, b, hq, D), (b, hkv, p0 + s, D), (b, hkv, p0 + s, D))))
    want, want_lse = orc.attention(q, k, v, D ** -0.5, dtype, position_index=p0)
    got, lse = gpu_attention(q, k, v, D ** -0.5, dtype, position_index=p0)
    res = compare(got, orc.from_storage(want, dtype), dtype)
    assert res["ok"], res
    assert float(np.abs(lse - want_lse).max()) <= LSE_TOL


@pytest.mark.parametrize("pieces,hs,b,hq,hkv,p0,s", OTHER, ids=_ids(OTHER))
def test_pieces_of_other_heads(pieces, hs, b, hq, hkv, p0, s):
    print("pieces", pieces, hs, b, hq, hkv, p0, s, flush=True)
    dtype = orc.BF16 if pieces % 2 else orc.F16
    assert plan_probe.general_plan(hs, 2, b, b, hq, hkv, p0, s)[:2] == ("chunk", pieces)
    q, k, v = (_rand(n, 620 + i, dtype) for i, n in enumerate(((s, b, hq, hs), (b, hkv, p0 + s, hs), (b, hkv, p0 + s, hs))))
    want, want_lse = orc.attention(q, k, v, hs ** -0.5, dtype, position_index=p0)
    got, lse = _run(q, k, v, hs ** -0.5, dtype, p0=p0)
    _check("%d pieces" % pieces, got, lse, want, want_lse, dtype, b)


def _late_score(hs, b, hq, hkv, p0, s, piece_keys, dtype):
    """One key 20 binary orders above all others, the first that every row sees or the chunk's first token in turn, its
    value zero; the other values such that a piece's sum is 1.49 to 1.5 x 2^127.  Any two added before they are weighted
    against that one pass binary32's range.  What was asked for, and the value and log-sum-exp of every row."""
    q, k = np.zeros((s, b, hq, hs), np.float32), np.zeros((b, hkv, p0 + s, hs), np.float32)
    q[..., 0] = 1.0
    value = np.array([1.5 * 2.0 ** 127 / piece_keys], np.float32)
    value = (value.view(np.uint32) & 0xffff0000).view(np.float32)[0]        # (eight bits: sums of up to 2^16 of them are exact)
    v = np.full(k.shape, value)
    for plane in range(b * hkv):
        hot = 0 if plane % 2 else p0
        k[plane // hkv, plane % hkv, hot, 0] = 20.0
        v[plane // hkv, plane % hkv, hot] = 0.0
    others = p0 + np.arange(s)
    total = others + 2.0 ** 20
    return *(orc.to_storage(x, dtype) for x in (q, k, v)), float(value) * others / total, np.log(total)


def _check_late_score(got, lse, want, want_lse, dtype):
    assert bool(np.isfinite(got).all())
    err = float(np.abs(got.astype(np.float64) / want[:, None, None, None] - 1.0).max())
    # A score of 20 in binary32 is off by up to 2^-20 (the scale's log2 and the product round once each), which is as
    # much of the weight; a piece's sum is exact, their fold and the division round a few times by 2^-24, and a 16-bit
    # output by half of its last place.
    assert err <= 2.0 ** -18 + (0.0 if dtype == orc.F32 else 2.0 ** -8), err
    assert np.abs(lse - want_lse[:, None, None]).max() <= LSE_TOL


@pytest.mark.parametrize("pieces,b,hq,hkv,p0,s", WIDE, ids=_ids(WIDE))
def test_large_values_under_a_late_score_wide(pieces, b, hq, hkv, p0, s):
    print("pieces", pieces, b, hq, hkv, p0, s, flush=True)
    call = (b, b, hq, hkv, p0, s)
    assert plan_probe.chunk_plan(*call, bf16=True)[2] == pieces
    q, k, v, want, want_lse = _late_score(D, b, hq, hkv, p0, s, plan_probe.chunk_piece_keys(*call, bf16=True), orc.BF16)
    got, lse = gpu_attention(q, k, v, float(np.log(2.0)), orc.BF16, position_index=p0)
    _check_late_score(got, lse, want, want_lse, orc.BF16)


@pytest.mark.parametrize("dtype", [orc.BF16, orc.F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("pieces,hs,b,hq,hkv,p0,s", OTHER, ids=_ids(OTHER))
def test_large_values_under_a_late_score_other(pieces, hs, b, hq, hkv, p0, s, dtype):
    print("pieces", pieces, hs, b, hq, hkv, p0, s, flush=True)
    plan = plan_probe.general_plan(hs, 4 if dtype == orc.F32 else 2, b, b, hq, hkv, p0, s)
    assert plan[0] == "chunk" and (plan[1] == pieces if dtype == orc.BF16 else plan[1] > 1)
    q, k, v, want, want_lse = _late_score(hs, b, hq, hkv, p0, s, plan[7], dtype)
    got, lse = _run(q, k, v, float(np.log(2.0)), dtype, p0=p0)
    _check_late_score(got, lse, want, want_lse, dtype)
