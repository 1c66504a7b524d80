"""Fused vector kernels of the Davidson iteration: blocks around a wave's four columns and at the
largest, dimensions around a workgroup's 64 rows, bases that restart with the corrections in columns
the same kernel reads (max_basis b + 1, 2 b, one short of 3 b), a basis as large as the operator, and
tolerances at which residuals reach rounding noise, so that blocks cannot be whitened by a Cholesky
factorisation. Eigenvalues lie within the residual tolerance of an eigenvalue of the oracle's matrix
(Hermitian) and rounding, 1e-12 of its norm; residuals of the returned vectors within twice the
tolerance; the vectors orthonormal to 1e-9 (a block is whitened at condition numbers to 1e6, times
2^-52 and the block)."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu

_H = {}


def operator(n):
    if n not in _H:
        ex = oracle_case(MODELS / "hBN.model", n, 1, 0, (1, 1, 10), exchange=True, Q=(0.02, 0.0, 0.0))
        _H[n] = (ex, ex.bse())
    return _H[n]


@pytest.mark.parametrize("n,nstates,block,max_basis,tol", [
    (3, 2, 3, 4, 1e-9), (3, 3, 9, 9, 1e-9), (4, 4, 8, 16, 1e-11), (6, 1, 1, 2, 1e-5), (6, 4, 5, 14, 1e-8),
    (6, 8, 8, 36, 1e-11), (8, 3, 4, 8, 1e-8), (8, 9, 31, 64, 1e-8), (9, 5, 13, 14, 1e-7), (12, 8, 32, 95, 1e-10),
    (12, 16, 32, 96, 1e-8), (13, 16, 17, 128, 1e-8)])
def test_solver_step(n, nstates, block, max_basis, tol):
    print(f"[step] N {n * n} states {nstates} block {block} basis {max_basis}", flush=True)
    ex, H = operator(n)
    ctx = gpu_context(ex)
    ctx.build(0)
    w, v, rep = ctx.solve(nstates=nstates, block=block, max_basis=max_basis, tol=tol, max_iter=3000)
    ctx.close()
    assert rep.converged
    ref = np.linalg.eigvalsh(H)
    assert max(np.abs(ref - e).min() for e in w) < tol + 1e-12 * np.abs(ref).max()
    assert np.linalg.norm(H @ v - v * w, axis=0).max() < 2 * tol + 1e-12 * np.abs(ref).max()
    assert np.abs(v.conj().T @ v - np.eye(nstates)).max() < 1e-9
