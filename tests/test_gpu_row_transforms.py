"""The convolution product on its row and column transforms: every kind of side they support (the
smallest and largest, square and uneven factor pairs, one factor equal to 1, long prime factors), windows narrower than
the mesh and as wide as it, reduced meshes (mesh points without a k-point), unequal band numbers,
and offsets that place two k-points on one mesh point (which stays on the general path). Reference:
the oracle's matrix; FP64 within 1e-12 and FP32 within 1e-5 of the largest entry of H X, as the other
product tests."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case, rel_err

pytestmark = pytest.mark.gpu


def check(ex, nvec, seed):
    H = ex.bse()
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(len(H), nvec)) + 1j * rng.normal(size=(len(H), nvec))
    ref = H @ x
    assert rel_err(ctx.matvec(x, precision=0, matrix_free=1), ref) < 1e-12
    assert rel_err(ctx.matvec(x, precision=1, matrix_free=1), ref) < 1e-5
    ctx.close()


@pytest.mark.parametrize("n", [2, 3, 5, 6, 8, 9, 10, 12, 15, 18, 20, 24, 25, 27, 30, 32, 36])
def test_sides(n):
    print(f"[rows] hBN {n}x{n}", flush=True)
    check(oracle_case(MODELS / "hBN.model", n, 1, 0, (1, 1, 10), cutoff=n / 3, exchange=True, Q=(0.03, 0, 0)), 3, n)


@pytest.mark.parametrize("n", [40, 54, 64, 75, 81, 90, 108, 120, 128])
def test_large_sides(n):
    # against the recomputed-tiles operator, which shares no code with the transforms
    print(f"[rows] hBN {n}x{n}", flush=True)
    ex = oracle_case(MODELS / "hBN.model", n, 1, 0, (1, 1, 10), cutoff=8, exchange=True)
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(n)
    x = rng.normal(size=(ex.N, 2)) + 1j * rng.normal(size=(ex.N, 2))
    ref = ctx.matvec(x, precision=0, matrix_free=2)
    assert rel_err(ctx.matvec(x, precision=0, matrix_free=1), ref) < 1e-12
    assert rel_err(ctx.matvec(x, precision=1, matrix_free=1), ref) < 1e-5
    ctx.close()


@pytest.mark.parametrize("n", [7, 11, 13, 14, 17, 19, 21, 22, 23, 26, 28, 29, 31, 33, 34, 35])
def test_sides_with_prime_factors(n):
    print(f"[rows] hBN {n}x{n}", flush=True)
    check(oracle_case(MODELS / "hBN.model", n, 1, 0, (1, 1, 10), cutoff=n / 3, exchange=True, Q=(0.03, 0, 0)), 3, n)


@pytest.mark.parametrize("n", [38, 46, 49, 57, 58, 62, 69, 77, 87, 91, 92, 93, 98, 102, 110, 112, 115, 119, 121, 124, 126, 37, 41,
                               43, 47, 53, 59, 61, 74, 106, 111, 122, 123, 67])
def test_large_sides_with_prime_factors(n):
    # against the recomputed-tiles operator, which shares no code with the transforms; from 43 on the
    # primes and their multiples stay on the transforms over whole meshes
    test_large_sides(n)


@pytest.mark.parametrize("n", [7, 13, 23])
@pytest.mark.parametrize("bands", [(1, 3), (3, 1), (4, 4)])
def test_bands_with_prime_factors(n, bands, synthetic18):
    nv, nc = bands
    print(f"[rows] {n}x{n} bands {bands}", flush=True)
    ex = oracle_case(synthetic18, n, 4, 0, (1, 1, 40), cutoff=2.0, exchange=True, bands=list(range(1 - nv, nc + 1)))
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(n)
    x = rng.normal(size=(ex.N, 2)) + 1j * rng.normal(size=(ex.N, 2))
    ref = ctx.matvec(x, precision=0, matrix_free=2)
    assert rel_err(ctx.matvec(x, precision=0, matrix_free=1), ref) < 1e-12
    assert rel_err(ctx.matvec(x, precision=1, matrix_free=1), ref) < 1e-5
    ctx.close()


@pytest.mark.parametrize("cutoff", [1.0, 3.0, 30.0])
@pytest.mark.parametrize("bands", [(1, 3), (3, 1), (4, 4)])
def test_windows_and_bands(cutoff, bands, synthetic18):
    nv, nc = bands
    print(f"[rows] window {cutoff} bands {bands}", flush=True)
    ex = oracle_case(synthetic18, 8, 4, 0, (1, 1, 40), cutoff=cutoff, exchange=True, Q=(0.0, 0.02, 0.0),
                     bands=list(range(1 - nv, nc + 1)))
    assert (ex.nv, ex.nc) == bands
    check(ex, 33, 7)


def test_reduced_mesh(synthetic18):
    print("[rows] reduced mesh", flush=True)
    check(oracle_case(synthetic18, 5, 2, 0, (1, 1, 40), factor=3, shift=(0.1, 0.2, 0), cutoff=2, exchange=True), 5, 11)


def test_shared_mesh_points():
    """Two k-points on one mesh point: the product is still defined by the matrix (the sum over k-points
    does not care), and the transforms, which hold one k-point per mesh point, must not take it."""
    print("[rows] shared mesh points", flush=True)
    ex = oracle_case(MODELS / "hBN.model", 6, 1, 0, (1, 1, 10), exchange=True)
    from xatu_amd import capi
    from cases import k_offsets
    s = ex.sys
    off = k_offsets(ex)
    off[1] = off[0] + [6, 0]
    ctx = capi.Context(0)
    ctx.set_lattice(s.bravais[:s.ndim], s.motif[:, :3], s.orb_per_atom, 6)
    ctx.set_bands(1, 1, ex.eigval_k, ex.eigvec_k, off, ex.eigval_kq, ex.eigvec_kq)
    ctx.fourier_sums(ex.eps_m, ex.eps_s, ex.r0, ex.cutoff, 6, ex.total_cells, exchange=True)
    ctx.build(2)
    x = np.zeros((ex.N, 1), complex)
    x[5] = 1.0  # a column away from the shared point: the rows of both k-points are defined
    y = ctx.matvec(x, precision=0, matrix_free=1)
    ref = ctx.matvec(x, precision=0, matrix_free=2)
    assert rel_err(y, ref) < 1e-12
    ctx.close()
