"""Contractions of the screening gradients: dimensions below, at and past one row per thread of the
exchange sums (256) and with runs that do not divide it, one to three atoms, Q that leaves V(Q) complex, with
and without exchange, more states than one pass of the transforms. For the Keldysh potential dH/d eps_s =
-(H - K) / (2 eps_bar), K the band energies on the diagonal, so psi^H dH psi follows from the built matrix
for any psi. Bound: sums of N^2 products, 1e-12 of the largest |psi|^H |H - K| |psi|."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,exchange,Q,states", [
    (1, True, (0, 0, 0), 1), (3, True, (0.05, 0.02, 0), 2), (15, True, (0.05, 0.02, 0), 9), (16, True, (0.1, 0, 0), 3),
    (17, True, (0.05, 0.02, 0), 8), (23, False, (0, 0, 0), 4), (43, True, (0.02, 0.03, 0), 2)])
@pytest.mark.parametrize("model", ["hBN", "synthetic18"])
def test_screening_gradients(n, exchange, Q, states, model, synthetic18):
    if model == "synthetic18" and n > 17:
        pytest.skip("the two-atom model covers the large dimensions")
    from xatu_amd import capi
    print(f"[gradients] {model} {n}x{n}", flush=True)
    path = MODELS / "hBN.model" if model == "hBN" else synthetic18
    ex = oracle_case(path, n, 1, 0, (1.5, 2.5, 10), cutoff=max(1.0, n / 3), exchange=exchange, Q=Q)
    ctx = gpu_context(ex)
    H = ctx.build(0, copy_out=True)
    nv, nc = ex.nv, ex.nc
    ek, ekq = np.asarray(ex.eigval_k), np.asarray(ex.eigval_kq)
    K = (ekq[nv:nv + nc, :].T[:, :, None] - ek[:nv, :].T[:, None, :]).ravel()
    D = H - np.diag(K)
    rng = np.random.default_rng(n)
    x = rng.normal(size=(len(H), states)) + 1j * rng.normal(size=(len(H), states))
    x /= np.linalg.norm(x, axis=0)
    g = ctx.hf_gradients(states, [capi.XATU_PARAM_EPS_S], eigvec=x)[:, 0]
    ctx.close()
    ref = -np.real(np.einsum("is,is->s", x.conj(), D @ x)) / (2 * 2.0)
    bound = 1e-12 * np.einsum("is,is->s", np.abs(x), np.abs(D) @ np.abs(x)).max()
    assert np.abs(g - ref).max() <= max(bound, 1e-15)
