"""The merge launch of split chunk calls: counts of pieces below, at and above what a lane takes at once and what lanes
share (one lane up to eight pieces or in large grids, eight lanes to 32, 64 lanes beyond), 128-wide heads and others.
Same oracle and bounds as tests/test_gpu_random_shapes.py and tests/test_gpu_general_heads.py."""
import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from gpu_util import D, LSE_TOL, compare, gpu_attention, rand_storage
from test_gpu_general_heads import _check, _rand, _run

pytestmark = pytest.mark.gpu

# pieces, batch, q heads, kv heads, position_index, interval
WIDE = [(5, 1, 16, 1, 2500, 33), (6, 1, 4, 4, 1700, 2), (9, 12, 4, 4, 3300, 2), (10, 1, 16, 1, 5000, 33), (16, 1, 4, 4, 5000, 2),
        (20, 1, 16, 1, 5000, 9), (29, 1, 4, 4, 9000, 2), (36, 1, 16, 1, 9000, 9)]
# pieces, head size, batch, q heads, kv heads, position_index, interval
OTHER = [(2, 64, 1, 8, 1, 600, 5), (3, 64, 1, 8, 1, 1100, 5), (4, 64, 1, 8, 1, 1700, 5), (5, 64, 1, 8, 1, 2500, 5),
         (9, 64, 1, 8, 1, 4200, 5), (16, 64, 2, 4, 4, 9000, 70), (18, 64, 1, 8, 1, 9000, 5)]


@pytest.mark.parametrize("pieces,b,hq,hkv,p0,s", WIDE, ids=["%d_pieces" % c[0] for c in WIDE])
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


@pytest.mark.parametrize("pieces,hs,b,hq,hkv,p0,s", OTHER, ids=["%d_pieces" % c[0] for c in OTHER])
def test_pieces_of_other_heads(pieces, hs, b, hq, hkv, p0, s):
    print("pieces", pieces, hs, b, hq, hkv, p0, s, flush=True)
    dtype = orc.BF16 if pieces % 2 else orc.F16
    assert plan_probe.general_plan(hs, 2, b, b, hq, hkv, p0, s)[:2] == ("chunk", pieces)
    q, k, v = (_rand(n, 620 + i, dtype) for i, n in enumerate(((s, b, hq, hs), (b, hkv, p0 + s, hs), (b, hkv, p0 + s, hs))))
    want, want_lse = orc.attention(q, k, v, hs ** -0.5, dtype, position_index=p0)
    got, lse = _run(q, k, v, hs ** -0.5, dtype, p0=p0)
    _check("%d pieces" % pieces, got, lse, want, want_lse, dtype, b)
