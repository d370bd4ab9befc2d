"""The 256 x 256 projection tiles whose last round is cut into halves (256 tokens x one head) or
quarters (128 tokens x one head), and one-head tiles walked in bands.  Same oracle and bound as tests/test_gpu_projection.py."""
import pytest

import oracle_lib as orc
from gpu_util import D, compare_ulps, rand_storage, to_dev, to_host
from test_gpu_projection import TILES_256X2, _path, _rope_table, _run_matmul3, _weights

pytestmark = pytest.mark.gpu


def _tail_parts(rows, heads):
    """Workgroups per tile of the last round: 1 (whole tiles), 2 or 4."""
    import torch

    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = (rows + 255) // 256 * ((heads + 1) // 2)
    last = tiles % n_cu
    if tiles <= n_cu or last == 0 or 2 * last > n_cu:
        return 1
    return 4 if 4 * last <= n_cu else 2


# (rows, K, q heads, kv heads, dtype, parts on 256 units): tiles beyond whole rounds
QKV = [
    (3200, 64, 39, 1, orc.F16, 4),     # 17 of 273: odd head count, second token halves without rows, one chunk of K
    (3201, 192, 39, 1, orc.BF16, 4),   # ... with one row
    (4100, 128, 32, 4, orc.F16, 2),    # 84 of 340: four rows in the last token tiles
    (5100, 64, 29, 2, orc.BF16, 2),    # 84 of 340: odd head count
    (4096, 64, 40, 4, orc.F16, 2),     # 128 of 384: the most that is cut
    (5800, 64, 29, 2, orc.F16, 1),     # 135 of 391: stay whole
]


@pytest.mark.parametrize("rows,k,hq,hkv,dtype,parts", QKV)
def test_matmul3_last_round(rows, k, hq, hkv, dtype, parts):
    heads = hq + 2 * hkv
    assert _path(rows, heads, k) == TILES_256X2 and _tail_parts(rows, heads) == parts
    hidden = rand_storage((rows, 1, k), 11, dtype)
    w = _weights(k, hq, hkv, dtype, 20)
    cap = rows + 8
    got, want = _run_matmul3(hidden, *w, _rope_table(cap, dtype), dtype, 1, hq, hkv, cap, 5, rows, 1)
    for name, g, x in zip("qkv", got, want):
        r = compare_ulps(g, x, dtype)
        assert r["ok"], (name, r)
    for cache in got[1:]:
        assert not cache[:, :, :5].any() and not cache[:, :, 5 + rows:].any()


@pytest.mark.parametrize("rows,k,heads,dtype,parts", [(8193, 64, 16, orc.F16, 4), (10753, 64, 16, orc.BF16, 2),
                                                       (4230, 128, 33, orc.F16, 4)])
def test_matmul_add_last_round(rows, k, heads, dtype, parts):
    import torch

    import ellm_amd

    assert _path(rows, heads, k) == TILES_256X2 and _tail_parts(rows, heads) == parts
    a = rand_storage((rows, 1, k), 51, dtype)
    w = rand_storage((heads * D, k), 52, dtype, scale=k ** -0.5)
    r = rand_storage((rows, 1, heads * D), 53, dtype)
    da, dw, dr = to_dev(a, dtype), to_dev(w, dtype), to_dev(r, dtype)
    op = ellm_amd.MatMulAdd(da, dw, dr, dr)   # in place
    op.run(0, rows, 1)
    torch.cuda.synchronize()
    res = compare_ulps(to_host(dr, dtype), orc.from_storage(orc.matmul_add(a, w, r, dtype, batch_size=1), dtype), dtype)
    assert res["ok"], res
    op.close()


@pytest.mark.parametrize("rows,heads,path", [(1601, 16, 1), (3200, 17, 2), (3841, 16, 2)])   # 13 tiles in bands of 4, 4, 4, 1; 16 in bands of 4
def test_matmul_add_bands(rows, heads, path):
    import torch

    import ellm_amd

    assert _path(rows, heads, 64) == path
    a = rand_storage((rows, 1, 64), 51, orc.F16)
    w = rand_storage((heads * D, 64), 52, orc.F16, scale=0.125)
    r = rand_storage((rows, 1, heads * D), 53, orc.F16)
    da, dw, dr = to_dev(a, orc.F16), to_dev(w, orc.F16), to_dev(r, orc.F16)
    out = torch.zeros_like(dr)
    op = ellm_amd.MatMulAdd(da, dw, dr, out)
    op.run(0, rows, 1)
    torch.cuda.synchronize()
    res = compare_ulps(to_host(out, orc.F16), orc.from_storage(orc.matmul_add(a, w, r, orc.F16, batch_size=1), orc.F16), orc.F16)
    assert res["ok"], res
    op.close()
