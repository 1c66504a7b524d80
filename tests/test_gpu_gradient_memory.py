"""Screening gradients of eight states at a size where their correlation buffer in one pass would be 8.6 GB: they
keep within the 4 GB of the products' passes (5 GiB with the other buffers), and each state's gradients are those of
a call for it alone (sums of the same terms in the same order up to the pass: 1e-12)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_passes():
    import torch
    from xatu_amd import capi
    n, norb, states = 128, 64, 8
    print(f"[gradient memory] {n}x{n}, {norb} orbitals, {states} states", flush=True)
    rng = np.random.default_rng(0)
    nk = n * n
    q, _ = np.linalg.qr(rng.normal(size=(nk, norb, 2)) + 1j * rng.normal(size=(nk, norb, 2)))
    vec = np.asfortranarray(np.moveaxis(q, 0, 2))
    val = np.asfortranarray(np.stack([-1.5 - rng.random(nk), 1.5 + rng.random(nk)]))
    off = np.stack(np.unravel_index(np.arange(nk), (n, n), order="F"), axis=1).astype(np.int32)
    ctx = capi.Context(0)
    ctx.set_lattice(2.5 * np.eye(3)[:2], np.array([[0.0, 0.0, 0.0], [1.1, 0.4, 0.0]]), [32, 32], n)
    ctx.set_bands(1, 1, val, vec, off)
    ctx.fourier_sums(1, 1, 10.0, 100.0, n, nk, exchange=True)  # every cell of the supercell: the window is the mesh
    ctx.build(capi.XATU_MATRIX_FREE)
    x = rng.normal(size=(nk, states)) + 1j * rng.normal(size=(nk, states))
    x /= np.linalg.norm(x, axis=0)
    params = [capi.XATU_PARAM_R0, capi.XATU_PARAM_EPS_S]
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    g = ctx.hf_gradients(states, params, eigvec=x)
    used = free - torch.cuda.mem_get_info()[0]
    alone = np.concatenate([ctx.hf_gradients(1, params, eigvec=x[:, i:i + 1]) for i in (0, 3, 4, 7)])
    ctx.close()
    assert used < 5 << 30, used
    assert np.abs(g[[0, 3, 4, 7]] - alone).max() <= 1e-12 * np.abs(g).max()
