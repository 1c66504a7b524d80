"""Full diagonalisation of matrices whose off-diagonal entries are so small that their squares underflow
(very large dielectric constants: entries of 1e-151 to 1e-169 beside energies of order one), on every number of
rows the reduction's kernels are compiled for and with the library's back-transformation. Bounds as in
test_gpu_tridiagonal.py: 4 n 2^-53 of the norm, vectors orthonormal to 4 n 2^-53."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,eps", [(4, 1e158), (8, 1e150), (8, 1e158), (8, 1e161), (8, 1e165), (18, 1e158), (25, 1e161), (34, 1e160)])
def test_small_off_diagonals(n, eps):
    print(f"[tridiagonal] N {n * n} dielectric constant {eps}", flush=True)
    ex = oracle_case(MODELS / "hBN.model", n, 1, 0, (eps, eps, 10), cutoff=3, exchange=True, Q=(0.02, 0.01, 0))
    ctx = gpu_context(ex)
    H = ctx.build(0, copy_out=True)
    w, v, _ = ctx.solve(method=0, nstates=0)
    ctx.close()
    N = len(H)
    ref = np.linalg.eigvalsh(H)
    norm = np.abs(ref).max()
    bound = 4 * N * 2.0 ** -53
    off = np.abs(H - np.diag(np.diag(H)))
    assert 0 < off.max() < 1e-140
    assert np.all(np.diff(w) >= 0) and np.abs(w - ref).max() <= bound * norm
    assert np.linalg.norm(H @ v - v * w, axis=0).max() <= bound * norm
    assert np.abs(v.conj().T @ v - np.eye(N)).max() <= bound
