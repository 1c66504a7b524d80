"""A mesh of one k-point: the convolution products and the gradients, whose transforms have length one, against the
oracle's matrix to the bars of the other product tests, with unequal band numbers and more vectors than a block."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bands", [(1, 1), (2, 2), (1, 3), (4, 4)])
def test_products(bands, synthetic18):
    nv, nc = bands
    print(f"[single point] bands {bands}", flush=True)
    ex = oracle_case(synthetic18, 1, 4, 0, (1, 1, 40), cutoff=1.0, exchange=True, Q=(0.03, 0, 0), bands=list(range(1 - nv, nc + 1)))
    H = ex.bse()
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(nc)
    x = rng.normal(size=(len(H), 33)) + 1j * rng.normal(size=(len(H), 33))
    for _ in range(2):
        assert rel_err(ctx.matvec(x, precision=0, matrix_free=1), H @ x) < 1e-12
        assert rel_err(ctx.matvec(x, precision=1, matrix_free=1), H @ x) < 1e-5
    ctx.close()


def test_gradients():
    from test_gpu_band_adjoint import reference
    print("[single point] gradients", flush=True)
    ex = oracle_case(MODELS / "hBN.model", 1, 1, 0, (1, 1, 20), exchange=True, Q=(0.03, 0.01, 0), cutoff=1)
    ctx = gpu_context(ex)
    ctx.build(2)
    psi = np.exp(1j * np.arange(3))[None, :].copy()  # three states: the transforms
    w, g = ctx.band_gradients(3, eigvec=psi)
    ctx.close()
    for i in range(3):
        wr, gr = reference(ex, psi[:, i].copy())
        assert np.abs(w[i] - wr).max() < 1e-12
        assert np.abs(g[i] - gr).max() <= 1e-12 * np.abs(gr).max()
