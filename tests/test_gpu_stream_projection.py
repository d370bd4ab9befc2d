"""The weight-streaming projection at the edges of its tiles: columns per workgroup that divide no head
(24, 40, 48) or need several rounds, K that is no multiple of the waves' chunks, 1 to 64 rows either
side of the token blocks.  Same oracle and bound as tests/test_gpu_projection.py."""
import numpy as np
import pytest

import oracle_lib as orc
from gpu_util import compare_ulps, rand_storage, to_dev, to_host
from test_gpu_fused_step import _check_against_oracle, _Layer
from test_gpu_projection import _rope_table, _run_matmul3, _weights

pytestmark = pytest.mark.gpu

# (rows, K, q heads, kv heads, dtype): columns a workgroup on 256 compute units
QKV = [
    (1, 1088, 3, 1, orc.F16),       # 8 columns; 17 chunks of K: one wave takes three, the others two
    (17, 1024, 20, 10, orc.BF16),   # 24 columns: workgroups across heads and across the key / value boundary
    (5, 1024, 48, 16, orc.F16),     # 40 columns
    (33, 1024, 32, 32, orc.BF16),   # 48 columns, three token blocks
    (49, 8192, 1, 1, orc.F16),      # four token blocks, sixteen chunks a wave
]


@pytest.mark.parametrize("rows,k,hq,hkv,dtype", QKV)
def test_matmul3_rows(rows, k, hq, hkv, dtype):
    hidden = rand_storage((1, rows + 1, k), 11, dtype)
    w = _weights(k, hq, hkv, dtype, 20)
    got, want = _run_matmul3(hidden, *w, _rope_table(16, dtype), dtype, rows + 1, hq, hkv, 16, 3, 1, rows)
    for name, g, x in zip("qkv", got, want):
        r = compare_ulps(g, x, dtype)
        assert r["ok"], (name, r)
    assert not got[0][:, rows:].any() and not got[1][rows:].any() and not got[2][rows:].any()


@pytest.mark.parametrize("rows,k,n,dtype", [(16, 1024, 128, orc.F16), (48, 1152, 8320, orc.BF16), (64, 4096, 2176, orc.F16),
                                            (3, 1024, 12416, orc.F16)])   # the last: two rounds of 32 columns
def test_matmul_add_rows(rows, k, n, dtype):
    import torch

    import ellm_amd

    a = rand_storage((1, rows, k), 51, dtype)
    w = rand_storage((n, k), 52, dtype, scale=k ** -0.5)
    r = rand_storage((1, rows, n), 53, dtype)
    out = torch.zeros((1, rows, n), dtype=to_dev(r, dtype).dtype, device="cuda")
    op = ellm_amd.MatMulAdd(to_dev(a, dtype), to_dev(w, dtype), to_dev(r, dtype), out)
    for _ in range(2):
        op.run(0, 1, rows)
    torch.cuda.synchronize()
    res = compare_ulps(to_host(out, dtype), orc.from_storage(orc.matmul_add(a, w, r, dtype, batch_size=rows), dtype), dtype)
    assert res["ok"], res
    op.close()


def test_fused_step_of_24_sequences_on_8192_wide_rows():
    """More than 16 rows on K above 4096 run fused too: rows bit for bit as the ordinary calls leave them."""
    batch, pos = 24, list(range(3, 27))
    layer = _Layer(orc.F16, batch, 2, 1, 40, 8192, seed=10)
    try:
        assert layer.qkv.attention_path(layer.attn, batch) == 1
        layer.reset()
        layer.qkv.run(9, 1, batch)
        layer.attn.run(9, 1, batch)
        plain = layer.snapshot()
        layer.reset()
        layer.qkv.run_with_attention(layer.attn, 9, batch)
        fused = layer.snapshot()
        for a, b in zip(plain[:3], fused[:3]):
            assert np.array_equal(a, b)
        _check_against_oracle(layer, fused, [9] * batch, batch)
    finally:
        layer.close()
