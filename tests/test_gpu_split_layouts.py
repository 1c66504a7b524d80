"""The split product at dimensions whose work items hold several row blocks a column chunk: row blocks that start
inside a chunk, diagonal chunks with blocks after the diagonal, ragged last chunks and blocks, on the presplit
matrix (equal band numbers) and on the FP32 one (1 valence and 2 conduction bands). Against the product with the FP64 matrix, to
the bar of the other tests of this product."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case, rel_err

pytestmark = pytest.mark.gpu


# N = 9216 and 9604: 36 and 38 row blocks (the last one of 132 rows), chunks of 3; 12996: 51, the last of
# 196 rows, chunks of 6; 8978 and 9248: 36 and 37, the last of 18 and 32 rows, chunks of 3
@pytest.mark.parametrize("n,bands", [(96, (1, 1)), (98, (1, 1)), (114, (1, 1)), (67, (1, 2)), (68, (1, 2))])
def test_products(n, bands, synthetic18):
    nv, nc = bands
    path = MODELS / "hBN.model" if nc == 1 else synthetic18
    print(f"[split layouts] N {n * n * nv * nc}", flush=True)
    ex = oracle_case(path, n, nc, 0, (1, 1, 10), cutoff=8, exchange=True, bands=None if nc == 1 else [0, 1, 2])
    assert (ex.nv, ex.nc) == bands
    ctx = gpu_context(ex)
    ctx.build(0)
    ctx.build(1)
    rng = np.random.default_rng(n)
    x = rng.normal(size=(ex.N, 35)) + 1j * rng.normal(size=(ex.N, 35))  # two vector blocks
    y0 = ctx.matvec(x, precision=0)
    y1 = ctx.matvec(x, precision=1)
    ctx.close()
    for j in range(35):
        assert rel_err(y1[:, j], y0[:, j]) < 1e-5, j
