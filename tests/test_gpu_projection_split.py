"""Projections of 65 to some hundred rows whose K several workgroups share: the sums of the pieces meet in a second
launch.  Rows that end inside a token tile, pieces of unequal length, odd head counts, sequences beyond batch_size,
per-sequence positions, a residual that is the output; then a call of fewer rows and one of whole tiles on the
same handle.  Same oracle and bound as tests/test_gpu_projection.py."""
import ctypes

import numpy as np
import pytest

import oracle_lib as orc
import plan_probe
from ellm_amd import _lib
from gpu_util import D, compare_ulps, rand_storage, to_dev, to_host
from test_gpu_projection import TILES_128, _path, _rope_table, _run_matmul3, _weights

pytestmark = pytest.mark.gpu


class _MatMulAddHandle(ctypes.Structure):   # struct ellm_matmul_add of project_api.hip
    _fields_ = [("d", _lib.MatMulAddDesc), ("device", ctypes.c_int), ("ws", ctypes.c_void_p), ("counters", ctypes.c_void_p),
                ("part", ctypes.c_void_p), ("part_floats", ctypes.c_size_t)]

# interval, pitch, batch, K, q heads, kv heads, position_index, dtype, (128-token blocks a tile, pieces, half heads)
QKV = [
    (65, 1, 1, 64 * 33, 1, 1, 3, orc.F16, (1, 7, 1)),      # 33 chunks in seven pieces, one token tile a quarter empty and a row beyond half
    (44, 3, 2, 64 * 40, 3, 1, 9, orc.BF16, (1, 8, 1)),     # 131 rows: a second tile of three; a sequence beyond batch_size
    (1, 100, 97, 2048, 32, 4, 40, orc.F16, (1, 4, 1)),     # one token for a hundred sequences
    (130, 1, 1, 8192, 52, 4, 0, orc.BF16, (2, 3, 0)),      # 256-token tiles, half of them empty
]


def _plan(rows, heads, k):
    plan = plan_probe.project_split(rows, heads, k)
    return plan[0], plan[1], plan[3]


@pytest.mark.parametrize("interval,pitch,batch,k,hq,hkv,p0,dtype,plan", QKV)
def test_matmul3_pieces(interval, pitch, batch, k, hq, hkv, p0, dtype, plan):
    rows, heads, cap = (interval - 1) * pitch + batch, hq + 2 * hkv, p0 + interval + 5
    print("rows", rows, "heads", heads, "K", k, flush=True)
    assert _path(rows, heads, k) == TILES_128 and _plan(rows, heads, k) == plan
    hidden = rand_storage((interval, pitch, k), 11, dtype)
    w = _weights(k, hq, hkv, dtype, 20)
    positions = None if interval > 1 else (np.arange(pitch) % (cap - 1)).astype(np.uint32)
    got, want = _run_matmul3(hidden, *w, _rope_table(cap, dtype), dtype, pitch, hq, hkv, cap, p0, interval, batch,
                             positions=positions)
    for name, g, x in zip("qkv", got, want):
        r = compare_ulps(g, x, dtype)
        assert r["ok"], (name, r)


@pytest.mark.parametrize("rows,heads,k,dtype,plan", [(79, 16, 4096, orc.F16, (1, 8, 1)), (480, 16, 64 * 61, orc.BF16, (1, 4, 0)), (385, 16, 64 * 63, orc.BF16, (2, 6, 0)),
                                                      (300, 12, 64 * 25, orc.F16, (1, 5, 1))])
def test_matmul_add_pieces(rows, heads, k, dtype, plan):
    import torch

    import ellm_amd

    print("rows", rows, "heads", heads, "K", k, flush=True)
    assert _path(rows, heads, k) == TILES_128 and _plan(rows, heads, k) == plan
    more = 128 * (256 // heads)       # whole tiles: a round of them
    assert _path(more, heads, k) == TILES_128 and plan_probe.project_split(more, heads, k)[1] == 1
    a = rand_storage((more, 1, k), 51, dtype)
    w = rand_storage((heads * D, k), 52, dtype, scale=k ** -0.5)
    r = rand_storage((more, 1, heads * D), 53, dtype)
    da, dw, dr = to_dev(a, dtype), to_dev(w, dtype), to_dev(r, dtype)
    op = ellm_amd.MatMulAdd(da, dw, dr, dr)   # in place
    for n in (rows, 20, more):
        dr.copy_(to_dev(r, dtype))
        op.run(0, n, 1)
        torch.cuda.synchronize()
        got = to_host(dr, dtype)
        some = slice(max(0, n - 400), n)
        res = compare_ulps(got[some], orc.from_storage(orc.matmul_add(a[some], w, r[some], dtype, batch_size=1), dtype), dtype)
        assert res["ok"], (n, res)
        assert np.array_equal(got[n:], orc.from_storage(r[n:], dtype))   # rows past the call are left alone
    op.close()


def test_a_handle_without_room_keeps_k_whole():
    """What a handle does that was made when memory was out: its room is taken away behind its back, then each call that
    shared K runs with K whole and gives what the oracle gives.  That the room was there, and how much, first."""
    import torch

    import ellm_amd

    heads, k, dtype = 16, 4096, orc.F16
    rows = 300
    a = rand_storage((rows, 1, k), 61, dtype)
    w = rand_storage((heads * D, k), 62, dtype, scale=k ** -0.5)
    r = rand_storage((rows, 1, heads * D), 63, dtype)
    da, dw, dr = to_dev(a, dtype), to_dev(w, dtype), to_dev(r, dtype)
    out = torch.empty_like(dr)
    want = orc.from_storage(orc.matmul_add(a, w, r, dtype, batch_size=1), dtype)
    op = ellm_amd.MatMulAdd(da, dw, dr, out)
    handle = _MatMulAddHandle.from_address(op._handle.value)
    room, = plan_probe.project_room(heads, k, rows, rows)
    assert handle.part_floats == room[0] > 0 and handle.part == handle.ws + 4 * heads * D * 64
    seen = []
    for part, floats in ((handle.part, room[0]), (None, 0)):
        handle.part, handle.part_floats = part, floats
        for n in (rows, 79):
            assert _plan(n, heads, k)[1] > 2
            out.fill_(float("nan"))
            op.run(0, n, 1)
            torch.cuda.synchronize()
            seen.append(to_host(out, dtype))
            res = compare_ulps(seen[-1][:n], want[:n], dtype)
            assert res["ok"], (n, part, res)
    op.close()
    # (another order of the sums: the second pass did not share K)
    assert not np.array_equal(seen[0], seen[2])
