"""The projection tiles over the length of K: chunk counts below, at and above what the three shapes request
ahead (two to four chunks of 64) and the period their weight operands run in (three chunks); rows that end
inside a tile; two rounds of 128-token tiles.  Same oracle and bound as tests/test_gpu_projection.py."""
import pytest

import oracle_lib as orc
from gpu_util import D, compare_ulps, rand_storage, to_dev, to_host
from test_gpu_projection import TILES_128, TILES_256X1, TILES_256X2, _path

pytestmark = pytest.mark.gpu

SHAPES = [(130, 3, TILES_128), (513, 96, TILES_128), (3000, 20, TILES_256X1), (4097, 17, TILES_256X2)]


@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("rows,heads,path", SHAPES, ids=["128", "128_two_rounds", "256x1", "256x2"])
def test_k_of_few_chunks(rows, heads, path, chunks):
    import torch

    import ellm_amd

    k, dtype = 64 * chunks, orc.BF16 if chunks % 2 else orc.F16
    assert _path(rows, heads, k) == path
    a = rand_storage((rows, 1, k), 61, dtype)
    w = rand_storage((heads * D, k), 62, dtype, scale=k ** -0.5)
    r = rand_storage((rows, 1, heads * D), 63, dtype)
    da, dw, dr = to_dev(a, dtype), to_dev(w, dtype), to_dev(r, dtype)
    out = torch.zeros_like(dr)
    op = ellm_amd.MatMulAdd(da, dw, dr, out)
    op.run(0, rows, 1)
    torch.cuda.synchronize()
    res = compare_ulps(to_host(out, dtype), orc.from_storage(orc.matmul_add(a, w, r, dtype, batch_size=1), dtype), dtype)
    assert res["ok"], res
    op.close()
