"""The Davidson solver's Rayleigh-Ritz kernel at the sizes where its parts change form: bases that grow
through one and two column blocks (64), through the chunks of its back-transformation (16) and the
padding of its recurrences (4), up to the largest basis, blocks from 1 to 32, degenerate pairs
(hBN) and the FP32 reduction of the mixed form. A Ritz value lies within the residual norm of an
eigenvalue, so the energies must be within the solver's tolerance of the oracle's."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu

TOL = 1e-7


@pytest.fixture(scope="module")
def operator():
    ex = oracle_case(MODELS / "hBN.model", 16, 1, 0, (1, 1, 10), cutoff=6)
    H = ex.bse()
    ctx = gpu_context(ex)
    ctx.build(0)
    ctx.build(1)
    yield ctx, np.linalg.eigvalsh(H)
    ctx.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nstates,block,basis", [(2, 2, 9), (2, 4, 17), (2, 3, 62), (2, 5, 66), (3, 7, 100), (4, 9, 127),
                                                 (6, 16, 128), (8, 31, 128), (16, 32, 64), (16, 32, 65), (16, 32, 97),
                                                 (32, 32, 128)])
def test_basis_sizes(operator, nstates, block, basis, precision):
    ctx, exact = operator
    print(f"[rayleigh-ritz] nstates {nstates} block {block} basis {basis} precision {precision}", flush=True)
    w, v, rep = ctx.solve(method=1, nstates=nstates, block=block, max_basis=basis, precision=precision, tol=TOL,
                          max_iter=2000)
    assert rep.converged == 1
    assert np.abs(w - exact[:nstates]).max() < TOL
    assert np.abs(v.conj().T @ v - np.eye(nstates)).max() < 1e-10
