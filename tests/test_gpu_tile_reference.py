"""The reference maximum of the tile kernel and the streaming chunk kernel: exponentials are taken against the one a row has until a lane's
sum of them passes 2^15 (2^8 in bfloat16), then the row's true maximum is looked for and its sums are rescaled.  Score
levels that stay below that step, pass it once, again and again, fall back and pass it in some rows of a
block only; whole rows and a key range in splits, whose later splits some rows see nothing of, both on 32x32x16 instructions
("whole", "split") and on 16x16x32."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from gpu_util import D, LSE_TOL, gpu_attention, rand_storage, storage_ulp

pytestmark = pytest.mark.gpu

# levels of successive 64-key tiles, in units of the score's log2: below binary16's step of 15, once past it,
# rising all along, falling, up and down
LEVELS = {"below": [0, 13, 14, 12], "once": [0, 0, 17, 17], "rising": [0, 16, 40, 300], "falling": [300, 30, 10, 0],
          "waves": [0, 40, -40, 60]}


@pytest.mark.parametrize("b,hq,hkv,s,p0,want_kernel,split", [
    (16, 32, 4, 49, 200, "pingpong", False), (26, 32, 4, 49, 200, "pingpong", False), (1, 8, 1, 70, 2400, "pingpong", True),
    (16, 32, 1, 13, 2600, "pingpong", True), (2, 8, 1, 13, 2400, "stream", True), (2, 8, 1, 45, 2400, "stream", True)],
    ids=["whole", "whole_26", "split", "split_16", "stream_13", "stream_45"])
@pytest.mark.parametrize("name", LEVELS)
@pytest.mark.parametrize("dtype", [orc.F16, orc.BF16], ids=["f16", "bf16"])
def test_scores_that_outgrow_the_reference(b, hq, hkv, s, p0, want_kernel, split, name, dtype):
    cap = p0 + s
    kernel, _, n_split = plan_probe.chunk_plan(b, b, hq, hkv, p0, s)[:3]
    assert kernel == want_kernel and (n_split > 1) == split
    if kernel == "pingpong":
        assert plan_probe.chunk_form(b, b, hq, hkv, p0, s) == ("wide" if p0 + s == 249 and b == 16 or b == 1 else "registers")
    scale = 1.0 / math.sqrt(D)
    q = orc.from_storage(rand_storage((s, b, hq, D), 5, dtype), dtype)
    k = orc.from_storage(rand_storage((b, hkv, cap, D), 6, dtype), dtype)
    v = rand_storage((b, hkv, cap, D), 7, dtype)
    q[..., 0] = 8.0 * (np.arange(s)[:, None, None] % 3 - 1)    # of three rows one rises, one falls, one stays
    level = np.array([LEVELS[name][(i // 64) % 4] for i in range(cap)], dtype=np.float32)
    k[..., 0] = level * np.float32(math.log(2.0) / (8.0 * scale))
    q, k = orc.to_storage(q, dtype), orc.to_storage(k, dtype)
    got, lse = gpu_attention(q, k, v, scale, dtype, position_index=p0)
    want, want_lse = orc.attention(q, k, v, scale, dtype, position_index=p0)
    want = orc.from_storage(want, dtype)
    # Every weight is rounded to the storage type once, by half of its last place: at most 2^-11 (2^-8) of
    # what the row's weights make of the values' magnitudes; both sides round the output once.  (A row
    # with few keys that count may cancel to far less than that, so no bound relative to the output.)
    mags = orc.to_storage(np.abs(orc.from_storage(v, dtype)), dtype)
    size = orc.from_storage(orc.attention(q, k, mags, scale, dtype, position_index=p0)[0], dtype)
    err, bound = np.abs(got - want), (2.0 ** -11 if dtype == orc.F16 else 2.0 ** -8) * size + storage_ulp(want, dtype)
    assert (err <= bound).all(), float((err / bound).max())
    # (a log-sum-exp of up to 208 is spaced 2^-16; the bound leaves it a dozen roundings)
    assert np.abs(lse - want_lse).max() <= LSE_TOL + 12 * 2.0 ** -16


@pytest.mark.parametrize("b,hq,hkv,s,p0,want_kernel,split", [
    (16, 32, 4, 49, 200, "pingpong", False), (26, 32, 4, 49, 200, "pingpong", False), (3, 32, 4, 600, 4060, "pingpong", False), (1, 8, 1, 70, 2400, "pingpong", True),
    (16, 32, 1, 13, 2600, "pingpong", True), (300, 8, 1, 13, 520, "stream", False), (2, 8, 1, 13, 2400, "stream", True), (2, 8, 1, 45, 2400, "stream", True)],
    ids=["whole", "whole_26", "whole_4660_keys", "split", "split_16", "stream_whole", "stream_13", "stream_45"])
@pytest.mark.parametrize("rise", [7.5, 14.0])
def test_large_bfloat16_values_under_rising_scores(b, hq, hkv, s, p0, want_kernel, split, rise):
    """A value of 2^115 under the one score that lies 7.5 or 14 binary orders above those before it, in another
    place of the key range for every head: a weight of 2^14 would carry it past binary32's range."""
    kernel, _, n_split = plan_probe.chunk_plan(b, b, hq, hkv, p0, s)[:3]
    assert kernel == want_kernel and (n_split > 1) == split
    q, k, v = (np.zeros(n, np.float32) for n in ((s, b, hq, D), (b, hkv, p0 + s, D), (b, hkv, p0 + s, D)))
    q[..., 0] = 1.0
    planes = b * hkv
    hot = (np.arange(planes) * 37 % (p0 - 110)).reshape(b, hkv) + 100
    for i in range(b):
        for h in range(hkv):
            k[i, h, hot[i, h], 0] = rise
            v[i, h, hot[i, h]] = 2.0 ** 115
    q, k, v = (orc.to_storage(a, orc.BF16) for a in (q, k, v))
    got, _ = gpu_attention(q, k, v, float(np.log(2.0)), orc.BF16, position_index=p0)
    share = 1.0 / (1.0 + (p0 + np.arange(s)) * 2.0 ** -rise)          # of the one key among the row's keys
    err = np.abs(got / (share[:, None, None, None] * 2.0 ** 115) - 1.0)
    assert err.max() <= 2.0 ** -8 + 2.0 ** -9                         # the weights rounded once, the output once
