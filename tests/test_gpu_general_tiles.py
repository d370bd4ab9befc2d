"""The kernels for other head sizes and binary32 at the edges of their tiles: rows per workgroup (1, 16,
64 and 128), keys per step and turn, padded head blocks, key splits and their folds, rows that are not
whole 16-byte pieces, values that are not finite.  Every case says which kernel it is there for
(general_plan.hpp).  Same oracle and bounds as tests/test_gpu_general_heads.py."""
import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from test_gpu_general_heads import _check, _rand, _run

pytestmark = pytest.mark.gpu

# (name, dtype, batch, q heads, kv heads, head size, capacity, position_index, interval)
CASES = [
    ("rows_32_step_kernel_two_tiles", orc.F16, 1, 16, 1, 64, 200, 130, 2),
    ("rows_33_chunk_kernel", orc.BF16, 2, 3, 1, 64, 256, 150, 11),
    ("rows_128_one_tile", orc.F16, 1, 4, 1, 96, 96, 64, 32),
    ("rows_129_two_tiles", orc.BF16, 1, 3, 1, 160, 150, 100, 43),
    ("keys_64_and_65", orc.F16, 1, 2, 1, 32, 65, 0, 65),
    ("h224_padded_to_256", orc.F16, 1, 2, 1, 224, 120, 5, 70),
    ("h192_key_split", orc.BF16, 1, 8, 1, 192, 1100, 1040, 5),
    ("h64_key_split_many_rows", orc.F16, 1, 8, 2, 64, 2100, 2000, 67),
    ("f32_h64_key_split", orc.F32, 1, 8, 2, 64, 1500, 1400, 40),
    ("f32_h256", orc.F32, 1, 2, 1, 256, 130, 20, 60),
    ("f32_h96_three_tiles", orc.F32, 1, 3, 1, 96, 140, 20, 100),
    ("h64_four_groups_of_64_rows", orc.BF16, 1, 4, 1, 64, 300, 100, 80),
    ("h96_four_groups_last_steps_uneven", orc.F16, 1, 2, 1, 96, 200, 70, 63),
    ("h32_four_groups_three_steps", orc.F16, 1, 2, 2, 32, 140, 60, 70),
    ("h120_four_groups", orc.F16, 1, 3, 1, 120, 290, 150, 90),
    ("h64_two_groups_two_a_unit", orc.F16, 5, 64, 64, 64, 200, 10, 129),
    ("h80_two_groups", orc.BF16, 3, 64, 64, 80, 200, 30, 131),
    ("h96_more_than_one_a_unit", orc.BF16, 5, 64, 64, 96, 180, 0, 135),
    ("h160_two_groups_one_step_left", orc.F16, 2, 4, 2, 160, 165, 0, 161),
    ("h64_order_turns", orc.BF16, 4, 32, 32, 64, 390, 0, 385),
    ("h64_four_groups_key_split", orc.F16, 1, 4, 1, 64, 1700, 1600, 40),
    ("h33_elements_one_by_one", orc.F16, 2, 4, 2, 33, 180, 30, 50),
    ("f32_h130_elements_one_by_one", orc.F32, 1, 4, 1, 130, 100, 3, 40),
    ("step_group_17", orc.F16, 1, 17, 1, 64, 400, 399, 1),
    ("step_group_40_h256", orc.BF16, 1, 40, 1, 256, 300, 299, 1),
    ("step_fold_of_33_splits", orc.F16, 1, 4, 1, 128 - 8, 2110, 2109, 1),
    ("step_f32_h256_splits", orc.F32, 2, 8, 1, 256, 1030, 1027, 1),
    ("step_f32_h32", orc.F32, 1, 2, 2, 32, 700, 650, 1),
    ("step_h5_splits", orc.BF16, 1, 3, 1, 5, 600, 599, 1),
    # binary32 chunks of more rows than the row kernel is taken for: every padded head, one and several splits
    ("f32_chunk_h20_one_block", orc.F32, 1, 32, 4, 20, 210, 0, 200),
    ("f32_chunk_h64", orc.F32, 2, 32, 32, 64, 160, 30, 130),
    ("f32_chunk_h33_any_place", orc.F32, 1, 64, 8, 33, 150, 0, 150),
    ("f32_chunk_h96_key_split", orc.F32, 2, 16, 2, 96, 1030, 1000, 30),
    ("f32_chunk_h128_order_turns", orc.F32, 4, 32, 8, 128, 164, 100, 64),
    ("f32_chunk_h130_any_place", orc.F32, 4, 32, 8, 130, 164, 100, 64),
    ("f32_chunk_h192", orc.F32, 1, 64, 8, 192, 150, 0, 150),
    ("f32_chunk_h256_key_split", orc.F32, 1, 8, 2, 256, 1440, 1400, 40),
    ("f32_chunk_h256", orc.F32, 4, 32, 8, 256, 164, 100, 64),
    # the row kernel: one turn of keys, one key more, the widest head, a prompt, heads narrower than a piece
    ("rows_16_keys", orc.F16, 2, 8, 2, 64, 20, 0, 16),
    ("rows_17_keys", orc.F32, 1, 16, 4, 250, 20, 16, 1),
    ("rows_16_keys_h250", orc.BF16, 1, 16, 4, 250, 20, 15, 1),
    ("rows_h1", orc.F16, 2, 2, 1, 1, 12, 7, 4),
    ("rows_h256_f32", orc.F32, 1, 4, 4, 256, 140, 33, 100),
    ("rows_h3_f32", orc.F32, 1, 6, 2, 3, 50, 0, 50),
    ("chunk_h5_narrower_than_a_piece", orc.F16, 1, 8, 2, 5, 300, 100, 150),
    ("chunk_h3_f32_narrower_than_a_piece", orc.F32, 1, 64, 8, 3, 150, 0, 150),
]
ON_ROWS = {"f32_h256", "f32_h96_three_tiles", "f32_h130_elements_one_by_one"}


def _kernel(name):
    """The kernel a case is there for: by its name, or the one it takes since short walks have one."""
    if name in ON_ROWS or name.startswith("rows_") and "kernel" not in name and "_tile" not in name:
        return "rows"
    return "step" if name.startswith("step") or "step_kernel" in name else "chunk"


def element_bytes(dtype):
    return 4 if dtype == orc.F32 else 2


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tile_edges(case):
    name, dtype, b, hq, hkv, hs, cap, p0, s = case
    print("case", name, flush=True)
    assert plan_probe.general_plan(hs, element_bytes(dtype), b, b, hq, hkv, p0, s)[0] == _kernel(name)
    q, k, v = _rand((s, b, hq, hs), 31, dtype), _rand((b, hkv, cap, hs), 32, dtype), _rand((b, hkv, cap, hs), 33, dtype)
    scale = -0.9 / np.sqrt(hs) if hs == 96 else 1.0 / np.sqrt(hs)   # (a negative scale once per type)
    want, want_lse = orc.attention(q, k, v, scale, dtype, position_index=p0)
    got, lse = _run(q, k, v, scale, dtype, p0=p0)
    _check(name, got, lse, want, want_lse, dtype, b)


# (head size, q heads, kv heads, position_index, interval): chunks and single-token steps, one and several splits
BINARY32 = [(128, 8, 8, 169, 16), (128, 32, 8, 0, 185), (64, 32, 8, 300, 100), (256, 64, 8, 0, 150), (128, 8, 2, 1400, 40),
            (128, 8, 8, 291, 1), (64, 8, 2, 1900, 1), (256, 4, 1, 700, 1), (100, 4, 4, 60, 1), (256, 4, 4, 60, 64)]


@pytest.mark.parametrize("case", BINARY32, ids=["h%d_%dq%dkv_%d+%d" % c for c in BINARY32])
def test_binary32_sums_stay_in_short_chains(case):
    """Error against 64-bit arithmetic.  Rounding of a score's sum, of its exponent's argument, of the
    exponential and of the weighted sum each add about 2^-24 to a row (2-norm): together 1.1e-7 to 1.7e-7
    here, and the bound is 2^-22.  One chain of sums over a head of 128 or 256 gave 2.6e-7 to 5.3e-7.  The last
    case runs row by row."""
    hs, hq, hkv, p0, s = case
    print("case", case, flush=True)
    kernel = "step" if s == 1 or s * hq // hkv <= 32 else "rows" if case == BINARY32[-1] else "chunk"
    assert plan_probe.general_plan(hs, 4, 1, 1, hq, hkv, p0, s)[0] == kernel
    cap = p0 + s
    q, k, v = _rand((s, 1, hq, hs), 51, orc.F32), _rand((1, hkv, cap, hs), 52, orc.F32), _rand((1, hkv, cap, hs), 53, orc.F32)
    scale = np.float32(1.0 / np.sqrt(hs))
    got, lse = _run(q, k, v, float(scale), orc.F32, p0=p0)
    want = np.empty((s, 1, hq, hs))
    for h in range(hq):
        kk, vv = k[0, h // (hq // hkv)].astype(np.float64), v[0, h // (hq // hkv)].astype(np.float64)
        sc = q[:, 0, h].astype(np.float64) @ kk.T * np.float64(scale)
        sc[np.arange(cap)[None, :] > p0 + np.arange(s)[:, None]] = -np.inf
        w = np.exp(sc - sc.max(axis=1, keepdims=True))
        want[:, 0, h] = w @ vv / w.sum(axis=1, keepdims=True)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("relative error %.3g" % err, flush=True)
    assert err <= 2.4e-7


@pytest.mark.parametrize("dtype,hq,hkv,hs,p0,s", [(orc.F16, 8, 2, 64, 100, 70), (orc.BF16, 8, 1, 192, 600, 9),
                                                   (orc.F32, 4, 1, 128, 40, 3)])
def test_values_beyond_a_row_are_not_seen(dtype, hq, hkv, hs, p0, s):
    """The value row of the chunk's last token holds infinities: rows of earlier tokens come out as if
    it were not there (chunk kernel unsplit and split, step kernel with several tokens)."""
    cap = p0 + s + 3
    q, k, v = _rand((s, 1, hq, hs), 41, dtype), _rand((1, hkv, cap, hs), 42, dtype), _rand((1, hkv, cap, hs), 43, dtype)
    scale = 1.0 / np.sqrt(hs)
    want, want_lse = orc.attention(q, k, v, scale, dtype, position_index=p0)
    v2 = v.copy()
    if dtype == orc.F32:
        v2[:, :, p0 + s - 1:] = np.inf
    else:
        v2.view(np.uint16)[:, :, p0 + s - 1:] = 0x7C00 if dtype == orc.F16 else 0x7F80
    got, lse = _run(q, k, v2, scale, dtype, p0=p0)
    _check("infinite_last_value", got[:-1], lse[:-1], want[:-1], want_lse[:-1], dtype, 1)
    assert np.isposinf(got[-1]).all() and np.abs(lse[-1] - want_lse[-1]).max() <= 1e-4


@pytest.mark.parametrize("dtype,hs", [(orc.F16, 64), (orc.BF16, 96), (orc.F16, 256)])
@pytest.mark.parametrize("p0", [31, 32, 33, 63, 64, 95, 127])
def test_one_value_beyond_a_row_at_the_edges_of_steps(dtype, hs, p0):
    """The chunk kernel looks at values only from the first step on whose keys its first row must not see: one infinite
    element, in either half of a register, in the value row right behind that row's position."""
    s, hq, hkv = 40, 4, 1
    q, k, v = (_rand(n, 71 + i, dtype) for i, n in enumerate(((s, 1, hq, hs), (1, hkv, p0 + s, hs), (1, hkv, p0 + s, hs))))
    print("p0", p0, "head", hs, flush=True)
    assert plan_probe.general_plan(hs, 2, 1, 1, hq, hkv, p0, s)[0] == "chunk"
    want, want_lse = orc.attention(q, k, v, hs ** -0.5, dtype, position_index=p0)
    for column in (0, hs - 1):
        v2 = v.copy()
        v2.view(np.uint16)[:, :, p0 + 1, column] = 0x7C00 if dtype == orc.F16 else 0x7F80
        got, lse = _run(q, k, v2, hs ** -0.5, dtype, p0=p0)
        _check("infinite_next_value", got[:1], lse[:1], want[:1], want_lse[:1], dtype, 1)
        assert np.isposinf(got[1:, ..., column]).all()
        keep = np.arange(hs) != column
        _check("other_columns", got[1:][..., keep], lse[1:], want[1:][..., keep], want_lse[1:], dtype, 1)


# (q heads, kv heads, head size, position_index, interval): chunk kernel with one, two and four key groups and with a
# key split, step kernel with one and several splits, several tokens
INFINITE = [(8, 8, 64, 20, 40), (8, 2, 64, 400, 40), (4, 4, 192, 300, 140), (8, 1, 96, 1500, 9), (4, 4, 80, 40, 1),
            (8, 1, 64, 1700, 1), (4, 2, 33, 90, 5)]


@pytest.mark.parametrize("dtype", [orc.F16, orc.BF16, orc.F32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", INFINITE, ids=["%dq%dkv_h%d_%d+%d" % c for c in INFINITE])
def test_an_infinite_value_that_a_row_sees(case, dtype):
    """Infinities of either sign in the value row of one key that every row sees (the weight is positive, so
    that is what comes out), and finite values beside them.  As two 16-bit operands the weight has a rest of
    zero or of either sign, and 0 x inf is not a number."""
    hq, hkv, hs, p0, s = case
    print("case", case, dtype, flush=True)
    cap = p0 + s + 2
    q, k, v = _rand((s, 1, hq, hs), 61, dtype), _rand((1, hkv, cap, hs), 62, dtype), _rand((1, hkv, cap, hs), 63, dtype)
    f = v.view(np.float32 if dtype == orc.F32 else np.uint16)
    plus = np.inf if dtype == orc.F32 else 0x7C00 if dtype == orc.F16 else 0x7F80
    minus = -np.inf if dtype == orc.F32 else plus | 0x8000
    f[:, :, 7, 0::3], f[:, :, 7, 1::3] = plus, minus
    scale = 1.0 / np.sqrt(hs)
    want, want_lse = orc.attention(q, k, v, scale, dtype, position_index=p0)
    got, lse = _run(q, k, v, scale, dtype, p0=p0)
    right = [int(np.isposinf(got[..., 0::3]).sum()), int(np.isneginf(got[..., 1::3]).sum())]
    assert right == [got[..., 0::3].size, got[..., 1::3].size]
    w = orc.from_storage(want, dtype)
    _check("finite_columns", got[..., 2::3], lse, orc.to_storage(np.ascontiguousarray(w[..., 2::3]), dtype), want_lse, dtype, 1)


@pytest.mark.parametrize("dtype,hs,hq", [(orc.BF16, 256, 4), (orc.BF16, 64, 4), (orc.F32, 64, 64)], ids=["bf16_h256", "bf16_h64", "f32_h64"])
@pytest.mark.parametrize("rise", [6.5, 14.0])
def test_large_finite_values_under_rising_scores(dtype, hs, hq, rise):
    """One value of 1e38 under the highest score, which lies 6.5 or 14 binary orders above those of the step of keys
    before it: less and more than what makes the chunk kernel move its reference (by 8), so the weight is 2^6.5
    or 1 there."""
    hkv, s, p0 = 2, 50, 90
    assert plan_probe.general_plan(hs, element_bytes(dtype), 1, 1, hq, hkv, p0, s)[0] == "chunk"
    q, k, v = np.zeros((s, 1, hq, hs), np.float32), np.zeros((1, hkv, p0 + s, hs), np.float32), np.zeros((1, hkv, p0 + s, hs), np.float32)
    q[..., 0] = 1.0
    k[:, :, 70, 0] = rise
    v[:, :, 70] = 1e38
    q, k, v = (orc.to_storage(a, dtype) for a in (q, k, v))
    got, _ = _run(q, k, v, float(np.log(2.0)), dtype, p0=p0)
    share = 1.0 / (1.0 + (p0 + np.arange(s)) * 2.0 ** -rise)          # of the one key among the row's keys
    want = share[:, None, None, None] * float(orc.from_storage(v, dtype).max())
    err = float(np.abs(got / want - 1.0).max())
    assert err <= (2.0 ** -8 if dtype == orc.BF16 else 1e-6)         # half a unit of bfloat16, binary32 sums


@pytest.mark.parametrize("dtype,hs", [(orc.F16, 33), (orc.F32, 256), (orc.BF16, 7)])
def test_row_kernel_with_a_position_per_sequence(dtype, hs):
    bcap, b, hq, hkv, cap = 4, 3, 8, 2, 30
    assert plan_probe.general_plan(hs, element_bytes(dtype), bcap, b, hq, hkv, 15, 1)[0] == "rows"
    q, k, v = _rand((1, bcap, hq, hs), 71, dtype), _rand((bcap, hkv, cap, hs), 72, dtype), _rand((bcap, hkv, cap, hs), 73, dtype)
    positions = [15, 0, 9]
    want, want_lse = orc.attention(q, k, v, 0.2, dtype, positions=np.array(positions + [0], dtype=np.uint32), batch=b)
    got, lse = _run(q, k, v, 0.2, dtype, batch=b, positions=positions)
    _check("rows_ragged", got, lse, want, want_lse, dtype, b)


def test_repeated_steps_fold_the_same_bits():
    """The arrival counters return to zero: the same handle launched many times gives the same bits."""
    import torch

    import ellm_amd

    b, hq, hkv, hs, cap = 2, 8, 2, 64, 3000
    q = torch.randn((1, b, hq, hs), device="cuda").to(torch.bfloat16)
    k = torch.randn((b, hkv, cap, hs), device="cuda").to(torch.bfloat16)
    v = torch.randn((b, hkv, cap, hs), device="cuda").to(torch.bfloat16)
    out = torch.zeros_like(q)
    op = ellm_amd.Attention(q, k, v, out, b, hq, hkv, hs, k.stride(), 0.125)
    op.run(cap - 1, 1, b)
    torch.cuda.synchronize()
    first = out.clone()
    for i in range(200):
        op.run(cap - 1 if i % 3 else cap // 2, 1, b)
    op.reset()
    out.zero_()
    op.run(cap - 1, 1, b)
    torch.cuda.synchronize()
    assert torch.equal(out, first)
    op.close()
