"""Mixed solves at the numbers of states where the block of the FP64 refinement changes its kind, with the
solver's own block: 26 to 33 around the limit of the device Rayleigh-Ritz kernel (32 vectors) with the convolution,
15 to 17 around a whole tile of 16 vectors with a resident FP64 matrix. Energies within the residual tolerance of
the eigenvalues of the built matrix."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.mark.parametrize("nstates,resident", [(26, False), (27, False), (31, False), (32, False), (33, False),
                                              (15, True), (16, True), (17, True), (32, True)])
def test_states(nstates, resident):
    from xatu_amd import capi
    print(f"[refinement] {nstates} states, FP64 matrix resident: {resident}", flush=True)
    rng = np.random.default_rng(nstates)
    n, norb = 18, 4
    nk = n * n
    q, _ = np.linalg.qr(rng.normal(size=(nk, norb, norb)) + 1j * rng.normal(size=(nk, norb, norb)))
    vec = np.asfortranarray(np.moveaxis(q[:, :, :2], 0, 2))  # orbital, band, k
    val = np.asfortranarray(np.stack([-1.5 - rng.random(nk), 1.5 + rng.random(nk)]))
    off = np.stack(np.unravel_index(np.arange(nk), (n, n), order="F"), axis=1).astype(np.int32)
    ctx = capi.Context(0)
    ctx.set_lattice(2.5 * np.eye(3)[:2], np.array([[0.0, 0.0, 0.0], [1.1, 0.4, 0.0]]), [2, 2], n)
    ctx.set_bands(1, 1, val, vec, off)
    ctx.fourier_sums(1, 1, 10.0, 4.0, n, nk, exchange=True)
    H = ctx.build(capi.XATU_FP64, copy_out=True)
    ctx.build(capi.XATU_FP32)
    if not resident:
        ctx.free_bse(capi.XATU_FP64)
    w, _, rep = ctx.solve(nstates=nstates, precision=capi.XATU_FP32, tol=TOL, want_vectors=False, max_iter=3000)
    ctx.close()
    assert rep.converged
    ref = np.linalg.eigvalsh(H)
    assert np.abs(w - ref[:nstates]).max() < TOL + 1e-12 * np.abs(ref).max()
