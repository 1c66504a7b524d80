"""Derivatives by the band data for one and two states on small meshes, where they come from the pairs of k-points,
and just past the sizes at which the transforms take over (512 and 32 mesh points times orbitals), against automatic
differentiation as in test_gpu_band_adjoint.py and to its bound."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case
from test_gpu_band_adjoint import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,nb,mesh,states", [
    ("hbn", 1, 1, 1), ("hbn", 1, 2, 1), ("hbn", 1, 4, 2), ("hbn", 1, 5, 2), ("hbn", 1, 5, 3), ("hbn", 1, 12, 1), ("hbn", 1, 16, 1),
    ("hbn", 1, 17, 1), ("synthetic18", 2, 5, 1), ("synthetic18", 2, 6, 1), ("synthetic36", 3, 2, 1)])
@pytest.mark.parametrize("exchange,Q", [(True, (0.03, 0.01, 0)), (False, (0, 0, 0))])
def test_few_states(model, nb, mesh, states, exchange, Q, synthetic18, synthetic36):
    print(f"[band adjoint] mesh {mesh} {model} {nb} states {states} exchange {exchange}", flush=True)
    path = {"hbn": MODELS / "hBN.model", "synthetic18": synthetic18, "synthetic36": synthetic36}[model]
    ex = oracle_case(path, mesh, nb, 0, (1, 1, 20), exchange=exchange, Q=Q, cutoff=min(2, mesh))
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(mesh)
    psi = rng.normal(size=(ex.N, states)) + 1j * rng.normal(size=(ex.N, states))
    psi /= np.linalg.norm(psi, axis=0)
    w, g = ctx.band_gradients(states, eigvec=psi)
    ctx.close()
    for i in range(states):
        wr, gr = reference(ex, psi[:, i].copy())
        assert np.abs(w[i] - wr).max() < 1e-12
        assert np.abs(g[i] - gr).max() < 1e-12 * np.abs(gr).max()
