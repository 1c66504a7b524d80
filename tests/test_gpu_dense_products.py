"""Products with the resident matrix over the vector blocks and sizes where their kernels change
form: blocks of at most 16 and of 32 vectors, partial last blocks, dimensions below and beside
the workgroups' rows, odd dimensions (FP32 matrix cores). Reference: the copied-out matrix times
the vectors in NumPy; tolerance for FP64 4 N eps relative to |H| |x| (a sum of N rounded complex
products), for the FP32 matrix 2^-20 (its products carry at least 22 bits)."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [3, 12, 13, 30, 31])
def test_vector_blocks(mesh):
    ex = oracle_case(MODELS / "hBN.model", mesh, 1, 0, (1, 1, 10), exchange=True, Q=(0.05, 0.0, 0.0))
    ctx = gpu_context(ex)
    H = ctx.build(0, copy_out=True)
    ctx.build(1)
    n = len(H)
    rng = np.random.default_rng(mesh)
    x = rng.normal(size=(n, 35)) + 1j * rng.normal(size=(n, 35))
    size = np.abs(H) @ np.abs(x)
    for nvec in (1, 7, 15, 16, 17, 31, 32, 33, 35):
        print(f"[dense products] N={n} vectors={nvec}", flush=True)
        ref = H @ x[:, :nvec]
        assert (np.abs(ctx.matvec(x[:, :nvec], precision=0) - ref) <= 4 * n * 2.3e-16 * size[:, :nvec]).all()
        assert (np.abs(ctx.matvec(x[:, :nvec], precision=1) - ref) <= 2.0 ** -20 * size[:, :nvec].max()).all()
    ctx.close()


@pytest.mark.parametrize("mesh", [8, 16, 20, 23])
def test_split_product_chunks(mesh, synthetic18):
    # the matrix stored split for the FP16 matrix cores (dimensions that are multiples of 32) or
    # as FP32 entries (23 x 23), one to several row blocks and column chunks of the product
    print(f"[split product] mesh {mesh}", flush=True)
    ex = oracle_case(synthetic18, mesh, 2, 0, (1, 1, 40), cutoff=8, exchange=True)
    ctx = gpu_context(ex)
    H = ctx.build(0, copy_out=True)
    ctx.build(1)
    n = len(H)
    rng = np.random.default_rng(mesh)
    x = rng.normal(size=(n, 33)) + 1j * rng.normal(size=(n, 33))
    size = np.abs(H) @ np.abs(x)
    for nvec in (1, 32, 33):
        y = ctx.matvec(x[:, :nvec], precision=1)
        assert (np.abs(y - H @ x[:, :nvec]) <= 2.0 ** -18 * size[:, :nvec].max()).all()
    ctx.close()
