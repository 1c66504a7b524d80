"""One context whose lattice is set again with another mesh, atoms, orbitals and bands alike: products and
gradients on the transforms over whole meshes (1-D meshes and sides without a factor pair), to a larger mesh,
to a smaller one and back, and between dimensions. Reference: the same calls on a fresh context, which run the
same kernels in the same order, hence equal results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lay(ctx, ndim, n, seed):
    rng = np.random.default_rng(seed)
    nk, norb = n ** ndim, 4
    tau = np.array([[0.0, 0.0, 0.0], [1.1, 0.4 * (ndim > 1), 0.0]])
    q, _ = np.linalg.qr(rng.normal(size=(nk, norb, norb)) + 1j * rng.normal(size=(nk, norb, norb)))
    vec = np.asfortranarray(np.moveaxis(q[:, :, :2], 0, 2))  # orbital, band, k
    val = np.asfortranarray(np.stack([-1.5 - rng.random(nk), 1.5 + rng.random(nk)]))
    off = np.stack(np.unravel_index(np.arange(nk), (n,) * ndim, order="F"), axis=1).astype(np.int32)
    ctx.set_lattice(2.5 * np.eye(3)[:ndim], tau, [2, 2], n)
    ctx.set_bands(1, 1, val, vec, off)
    ctx.fourier_sums(1, 1, 10.0, n / 3, n, nk, exchange=True)
    ctx.build(2)
    return nk


def results(ctx, N, seed):
    from xatu_amd import capi
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(N, 3)) + 1j * rng.normal(size=(N, 3))
    x /= np.linalg.norm(x, axis=0)
    out = [ctx.matvec(x, precision=p, matrix_free=1) for p in (0, 1)]
    out += [ctx.hf_gradients(3, [capi.XATU_PARAM_R0, capi.XATU_PARAM_EPS_M], eigvec=x), *ctx.band_gradients(3, eigvec=x)]
    return out, ctx.matvec(x, precision=0, matrix_free=2)


@pytest.mark.parametrize("meshes", [[(1, 90), (1, 60), (1, 90)], [(1, 43), (1, 97)], [(2, 43), (2, 47), (2, 43)],
                                    [(1, 43), (2, 43), (1, 43)], [(2, 43), (2, 12), (2, 43)]])
def test_set_lattice_again(meshes):
    from xatu_amd import capi
    ctx = capi.Context(0)
    for i, (ndim, n) in enumerate(meshes):
        print(f"[mesh change] {ndim}-D {n}", flush=True)
        got, tiles = results(ctx, lay(ctx, ndim, n, i), i)
        fresh = capi.Context(0)
        ref, _ = results(fresh, lay(fresh, ndim, n, i), i)
        fresh.close()
        # against the recomputed tiles, which take no transforms
        assert np.abs(got[0] - tiles).max() < 1e-12 * np.abs(tiles).max()
        for a, b in zip(got[:3], ref[:3]):
            assert np.array_equal(a, b)
        # the pairs of k-points add with atomics in any order: N terms of one scale
        for a, b in zip(got[3:], ref[3:]):
            assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    ctx.close()
