"""Derivatives of exciton energies by the band data on both of their paths (row and column transforms;
pairs of k-points where the mesh side has no factor pair), against automatic differentiation of
E = psi^H H psi, H written out from the oracle's lattice sums and the band vectors in 64 bits.
Tolerance 1e-12 of the largest derivative: sums of N rounded terms of one scale, N < 1000."""
import numpy as np
import pytest
import torch

from cases import MODELS, gpu_context, k_offsets, oracle_case

pytestmark = pytest.mark.gpu


def reference(ex, psi):
    """(w, g) as xatu_band_gradients lays them out, for one state."""
    s = ex.sys
    n, na = ex.ncell * s.factor, len(s.orb_per_atom)
    nk, nv, nc = ex.eigval_k.shape[1], ex.nv, ex.nc
    begin = np.concatenate([[0], np.cumsum(s.orb_per_atom)])
    C = torch.from_numpy(np.ascontiguousarray(ex.eigvec_kq[:, nv:].transpose(2, 1, 0))).requires_grad_(True)
    V = torch.from_numpy(np.ascontiguousarray(ex.eigvec_k[:, :nv].transpose(2, 1, 0))).requires_grad_(True)
    e = (torch.from_numpy(ex.eigval_kq[nv:].T[:, :, None] - ex.eigval_k[:nv].T[:, None, :])).requires_grad_(True)
    off = k_offsets(ex)
    d = (off[None] - off[:, None] + n // 2) % n
    at = torch.from_numpy((d * (n ** np.arange(d.shape[-1]))).sum(-1)).long()
    M = torch.from_numpy(np.ascontiguousarray(ex.ft))
    MQ = torch.from_numpy(np.ascontiguousarray(ex.ftq))
    F = torch.zeros((nk, nc, nv, nk, nc, nv), dtype=torch.complex128)
    rho = []
    for a in range(na):
        o = slice(begin[a], begin[a + 1])
        rho.append(torch.einsum("kci,kvi->kcv", C[:, :, o].conj(), V[:, :, o]).reshape(-1))
        rc = torch.einsum("kci,ldi->kcld", C[:, :, o].conj(), C[:, :, o])
        for b in range(na):
            p = slice(begin[b], begin[b + 1])
            rv = torch.einsum("lwi,kvi->kvlw", V[:, :, p].conj(), V[:, :, p])
            F = F + torch.einsum("kcld,kl,kvlw->kcvldw", rc, M[a, b][at], rv)
    F = F.reshape(nk * nc * nv, -1)
    if ex.exchange:
        E1 = torch.stack(rho)
        F = F - E1.T @ (MQ @ E1.conj())
    x = torch.from_numpy(psi)
    p = x.conj()[:, None] * x[None]
    upper = torch.triu(p * F, 1).sum()
    diag = (torch.diagonal(F).real * (x.abs() ** 2)).sum()
    (((x.abs() ** 2) * e.reshape(-1)).sum() - 2 * upper.real - diag).backward()
    w = np.zeros((2, nk, nv + nc))
    g = np.zeros((2, nk, nv + nc, C.shape[2]), complex)
    w[1, :, nv:] = e.grad.sum(2).numpy()
    w[0, :, :nv] = -e.grad.sum(1).numpy()
    g[1, :, nv:] = C.grad.numpy() / 2
    g[0, :, :nv] = V.grad.numpy() / 2
    return w, g


@pytest.mark.parametrize("exchange,Q", [(True, (0.03, 0.01, 0)), (True, (0, 0, 0)), (False, (0.02, 0, 0))])
@pytest.mark.parametrize("model,nb", [("hbn", 1), ("synthetic18", 1), ("synthetic18", 2), ("synthetic36", 3)])
@pytest.mark.parametrize("mesh,factor", [(5, 1), (6, 1), (7, 1), (5, 2)])
def test_band_gradients(mesh, model, nb, exchange, Q, factor, synthetic18, synthetic36):
    print(f"[band adjoint] mesh {mesh} {model} {nb} exchange {exchange} factor {factor}", flush=True)
    path = {"hbn": MODELS / "hBN.model", "synthetic18": synthetic18, "synthetic36": synthetic36}[model]
    ex = oracle_case(path, mesh, nb, 0, (1, 1, 20), exchange=exchange, Q=Q, factor=factor, cutoff=2)
    ctx = gpu_context(ex)
    ctx.build(2)
    rng = np.random.default_rng(mesh)
    ns = 9
    psi = rng.normal(size=(ex.N, ns)) + 1j * rng.normal(size=(ex.N, ns))
    psi /= np.linalg.norm(psi, axis=0)
    w, g = ctx.band_gradients(ns, eigvec=psi)
    for i in (0, 7, 8):
        wr, gr = reference(ex, psi[:, i].copy())
        assert np.abs(w[i] - wr).max() < 1e-12
        assert np.abs(g[i] - gr).max() < 1e-12 * np.abs(gr).max()
    ctx.close()
