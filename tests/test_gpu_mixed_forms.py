"""Mixed solves whose FP64 refinement runs on each form of the product: the convolution on row and
column transforms, over whole meshes (a side without a factor pair) and in one dimension, recomputed tiles
in two and three dimensions (where no convolution exists) and in the reciprocal mode, a resident FP64 matrix.
Energies within the residual tolerance of the eigenvalues of the built FP64 matrix."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.mark.parametrize("ndim,n,form,mode,both", [
    (2, 12, 1, 0, False), (2, 43, 1, 0, False), (1, 90, 1, 0, False), (2, 12, 2, 0, False), (3, 5, 2, 0, False),
    (3, 5, 0, 0, True), (2, 10, 1, 1, False), (2, 10, 0, 1, False), (2, 12, 0, 0, True), (2, 12, 0, 0, False)])
@pytest.mark.parametrize("nstates", [1, 5])
def test_refinement(ndim, n, form, mode, both, nstates):
    from xatu_amd import capi
    print(f"[mixed] {ndim}-D {n} form {form} mode {mode} both {both} states {nstates}", flush=True)
    rng = np.random.default_rng(ndim * 100 + n)
    nk, norb = n ** ndim, 4
    bravais = 2.5 * np.eye(3)[:ndim]
    tau = np.array([[0.0, 0.0, 0.0], [1.1, 0.4 * (ndim > 1), 0.3 * (ndim > 2)]])
    q, _ = np.linalg.qr(rng.normal(size=(nk, norb, norb)) + 1j * rng.normal(size=(nk, norb, norb)))
    vec = np.asfortranarray(np.moveaxis(q[:, :, :2], 0, 2))  # orbital, band, k
    val = np.asfortranarray(np.stack([-1.5 - rng.random(nk), 1.5 + rng.random(nk)]))
    off = np.stack(np.unravel_index(np.arange(nk), (n,) * ndim, order="F"), axis=1).astype(np.int32)
    ctx = capi.Context(0)
    ctx.set_lattice(bravais, tau, [2, 2], n)
    ctx.set_bands(1, 1, val, vec, off)
    ctx.fourier_sums(1, 1, 10.0, max(1.0, min(4.0, n / 3)), n, nk, exchange=mode == 0, mode=mode, n_reciprocal=3)
    H = ctx.build(capi.XATU_FP64, copy_out=True)
    if form:
        ctx.build(capi.XATU_MATRIX_FREE)
    else:
        ctx.build(capi.XATU_FP32)
    if not both:
        ctx.free_bse(capi.XATU_FP64)
    w, _, rep = ctx.solve(nstates=nstates, precision=capi.XATU_FP32, matrix_free=form, tol=TOL, want_vectors=False,
                          max_iter=3000)
    ctx.close()
    assert rep.converged
    ref = np.linalg.eigvalsh(H)
    assert np.abs(w - ref[:nstates]).max() < TOL + 1e-12 * np.abs(ref).max()
