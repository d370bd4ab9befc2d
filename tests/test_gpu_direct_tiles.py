"""The tile kernel's form that fetches K and V straight into LDS (unsplit walks of 4096 keys and more): last tiles
whole and ragged, rows past the last token, unusual scales, score levels that move a row's reference maximum, and
what lies beyond a row's position.  Against float64 attention of the same storage values."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from gpu_util import D, LSE_TOL, gpu_attention, rand_storage, storage_ulp, to_dev
from test_gpu_tile_reference import LEVELS

pytestmark = pytest.mark.gpu

# (sequences, query heads, key-value heads, tokens, position of the first)
SHAPES = {"last_tile_of_1": (25, 64, 1, 7, 4090), "whole_tiles": (25, 64, 1, 9, 4087), "two_row_blocks": (25, 32, 4, 49, 4060),
          "chunk_of_600": (3, 32, 4, 600, 4060)}


def _shape(name):
    b, hq, hkv, s, p0 = SHAPES[name]
    assert plan_probe.chunk_is_direct(b, b, hq, hkv, p0, s)
    return b, hq, hkv, s, p0


def _exact(q, k, v, scale, dtype, p0):
    """(outputs, log-sum-exps, weighted sums of |v|, the same with every weight cut to 2^-25 of the row's largest) in
    float64, and the largest sum |q| |k| of a score"""
    import torch

    q, k, v = (to_dev(a, dtype).double() for a in (q, k, v))
    s, b, hq, _ = q.shape
    hkv, keys = k.shape[1], p0 + s
    group = hq // hkv
    out, size, tiny = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
    lse = torch.empty((s, b, hq), dtype=torch.float64, device="cuda")
    masked = torch.arange(keys, device="cuda")[None, :] > p0 + torch.arange(s, device="cuda")[:, None]
    largest = 0.0
    for i in range(b):
        for h in range(hkv):
            kt, vs = k[i, h, :keys].t().contiguous(), v[i, h, :keys]
            for n in range(h * group, (h + 1) * group):
                rows = q[:, i, n].contiguous()
                score = (rows @ kt * scale).masked_fill(masked, -math.inf)
                lse[:, i, n] = torch.logsumexp(score, dim=1)
                w = torch.exp(score - lse[:, i, n, None])
                out[:, i, n], size[:, i, n] = w @ vs, w @ vs.abs()
                tiny[:, i, n] = torch.minimum(w, 2.0 ** -25 * w.amax(dim=1, keepdim=True)) @ vs.abs()
                largest = max(largest, float((rows.abs() @ kt.abs()).max()))
    return *(t.cpu().numpy() for t in (out, lse, size, tiny)), largest


def _check(q, k, v, scale, dtype, p0):
    got, lse = gpu_attention(q, k, v, scale, dtype, position_index=p0)
    want, want_lse, size, tiny, largest = _exact(q, k, v, scale, dtype, p0)
    # A weight is rounded to the storage type once, by half of its last place, in binary16 by up to 2^-25 of the row's
    # largest (but no more than itself) where it is below that type's normal numbers; a score is a chain of at most sixteen
    # binary32 roundings, each of no more than the sum of its products' magnitudes; the output is rounded once.
    weight = (2.0 ** -11 if dtype == orc.F16 else 2.0 ** -8) + 16 * 2.0 ** -24 * largest * abs(scale)
    err, bound = np.abs(got - want), weight * size + storage_ulp(want, dtype)
    if dtype == orc.F16:
        bound += tiny
    assert (err <= bound).all(), float((err / bound).max())
    # (a log-sum-exp of up to 208 is spaced 2^-16: a dozen roundings)
    assert np.abs(lse - want_lse).max() <= LSE_TOL + 12 * 2.0 ** -16


@pytest.mark.parametrize("scale", [0.09, -0.07, 0.0, 1.0])
@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("dtype", [orc.F16, orc.BF16], ids=["f16", "bf16"])
def test_edges_and_scales(dtype, name, scale):
    b, hq, hkv, s, p0 = _shape(name)
    q, k, v = (rand_storage(n, i, dtype) for i, n in enumerate(((s, b, hq, D), (b, hkv, p0 + s, D), (b, hkv, p0 + s, D))))
    _check(q, k, v, scale, dtype, p0)


@pytest.mark.parametrize("levels", LEVELS)
@pytest.mark.parametrize("name", ["last_tile_of_1", "two_row_blocks"])
@pytest.mark.parametrize("dtype", [orc.F16, orc.BF16], ids=["f16", "bf16"])
def test_scores_that_outgrow_the_reference(dtype, name, levels):
    b, hq, hkv, s, p0 = _shape(name)
    scale = 1.0 / math.sqrt(D)
    q = orc.from_storage(rand_storage((s, b, hq, D), 5, dtype), dtype)
    k = orc.from_storage(rand_storage((b, hkv, p0 + s, D), 6, dtype), dtype)
    v = rand_storage((b, hkv, p0 + s, D), 7, dtype)
    q[..., 0] = 8.0 * (np.arange(s)[:, None, None] % 3 - 1)    # of three rows one rises, one falls, one stays
    level = np.array([LEVELS[levels][(i // 64) % 4] for i in range(p0 + s)], dtype=np.float32)
    k[..., 0] = level * np.float32(math.log(2.0) / (8.0 * scale))
    _check(orc.to_storage(q, dtype), orc.to_storage(k, dtype), v, scale, dtype, p0)


@pytest.mark.parametrize("name", ["last_tile_of_1", "whole_tiles", "two_row_blocks"])
def test_what_lies_beyond_the_position_is_never_read(name):
    """NaN, infinities and large values behind the call's last position, an output buffer that holds infinities."""
    b, hq, hkv, s, p0 = _shape(name)
    cap = p0 + s + 200
    q, k, v = (rand_storage(n, 19 + i, orc.F16) for i, n in enumerate(((s, b, hq, D), (b, hkv, cap, D), (b, hkv, cap, D))))
    clean = gpu_attention(q, k, v, 0.09, orc.F16, position_index=p0)
    bad = np.array([0x7e00, 0x7c00, 0xfc00, 0x7bff], dtype=np.uint16)      # NaN, +Inf, -Inf, 65504
    for i, a in enumerate((k, v)):
        a[:, :, p0 + s:] = bad[(np.arange(a[:, :, p0 + s:].size) + i) % 4].reshape(a[:, :, p0 + s:].shape)
    dirty = gpu_attention(q, k, v, 0.09, orc.F16, position_index=p0, out_fill=float("inf"))
    assert np.array_equal(clean[0], dirty[0]) and np.array_equal(clean[1], dirty[1])


@pytest.mark.parametrize("name", ["last_tile_of_1", "two_row_blocks", "chunk_of_600"])
def test_finite_rows_of_later_tokens_change_no_bit(name):
    b, hq, hkv, s, p0 = _shape(name)
    cap, cut = p0 + s + 5, s // 2
    q, k, v = (rand_storage(n, 91 + i, orc.F16) for i, n in enumerate(((s, b, hq, D), (b, hkv, cap, D), (b, hkv, cap, D))))
    base = gpu_attention(q, k, v, 0.09, orc.F16, position_index=p0)
    k.view(np.float16)[:, :, p0 + cut:p0 + s] = 60000.0
    v.view(np.float16)[:, :, p0 + cut:p0 + s] = -65504.0
    pert = gpu_attention(q, k, v, 0.09, orc.F16, position_index=p0)
    for x, y in zip(base, pert):
        assert np.array_equal(x[:cut], y[:cut]) and not np.array_equal(x[cut:], y[cut:])


def test_causality_of_a_long_prompt():
    """Rows before position 4100 do not see the keys from there on; those from there on do."""
    s, cut = 4150, 4100
    assert plan_probe.chunk_is_direct(1, 1, 32, 4, 0, s)
    q, k, v = (rand_storage(n, 22 + i, orc.F16) for i, n in enumerate(((s, 1, 32, D), (1, 4, s, D), (1, 4, s, D))))
    base = gpu_attention(q, k, v, 0.09, orc.F16)[0]
    k[:, :, cut:], v[:, :, cut:] = (rand_storage((1, 4, s - cut, D), 25 + i, orc.F16) for i in range(2))
    pert = gpu_attention(q, k, v, 0.09, orc.F16)[0]
    assert np.array_equal(base[:cut], pert[:cut]) and not (base[cut:] == pert[cut:]).all(axis=-1).any()
