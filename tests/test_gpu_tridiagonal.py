"""Full diagonalisation on the own reduction to tridiagonal form and back-transformation (to 1024): dimensions around a wave's 64 rows,
the row counts its kernels are compiled for (256, 512, 1024, 2048), the smallest it takes (4 here) and one
past it, which stays with the library; real matrices without an exchange term among them, degenerate pairs
and off-diagonals that vanish. Errors of a backward stable reduction grow at most like n 2^-53 of the norm:
eigenvalues and residuals within 4 n 2^-53 |H|, vectors orthonormal to 4 n 2^-53."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nv,nc,cutoff,exchange", [
    (2, 1, 1, 1.0, True), (3, 1, 1, 1.0, False), (8, 1, 1, 3.0, True), (9, 1, 1, 3.0, True), (16, 1, 1, 6.0, False),
    (17, 1, 1, 6.0, True), (22, 1, 1, 8.0, True), (23, 1, 1, 8.0, False), (32, 1, 1, 10.0, True), (33, 1, 1, 0.5, True),
    (45, 1, 1, 8.0, True), (46, 1, 1, 2.0, False)])
def test_full_spectrum(n, nv, nc, cutoff, exchange):
    print(f"[tridiagonal] N {n * n * nv * nc}", flush=True)
    ex = oracle_case(MODELS / "hBN.model", n, 1, 0, (1, 1, 10), cutoff=cutoff, exchange=exchange, Q=(0.02, 0.01, 0))
    ctx = gpu_context(ex)
    H = ctx.build(0, copy_out=True)
    w, v, _ = ctx.solve(method=0, nstates=0)
    ctx.close()
    N = len(H)
    ref = np.linalg.eigvalsh(H)
    norm = np.abs(ref).max()
    bound = 4 * N * 2.0 ** -53
    assert len(w) == N and np.all(np.diff(w) >= 0)
    assert np.abs(w - ref).max() <= bound * norm
    assert np.linalg.norm(H @ v - v * w, axis=0).max() <= bound * norm
    assert np.abs(v.conj().T @ v - np.eye(N)).max() <= bound
