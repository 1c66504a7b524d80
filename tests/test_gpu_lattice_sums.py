"""Lattice Fourier sums of the mesh, taken over the rows of cells and then along them: sides around
the workgroup's width, odd and even, one cell, rows cut short by the cutoff, one to many atoms (the
row sums are held for a bounded number of pairs at a time). Reference: the two matrix products with
the roots of unity in NumPy, FP64. The bound is that of the reference's own recursive sums, (cells of
a row + rows + 16) 2^-53 of the sum of |V|; 16 covers the potential and the roots."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PREF = 1.6021766e-19 / (4e-10 * 3.141592653589793 * 8.8541878e-12)


@pytest.mark.parametrize("n,natoms,ncell,cutoff,angle", [
    (1, 1, 1, 0.3, 90), (2, 2, 4, 1.4, 60), (3, 1, 5, 1.6, 120), (24, 2, 24, 8.3, 60), (127, 3, 60, 23.7, 75),
    (128, 1, 31, 99.0, 60), (129, 2, 40, 12.1, 120), (300, 4, 21, 6.4, 60), (512, 10, 300, 80.2, 60)])
def test_mesh_sums(n, natoms, ncell, cutoff, angle):
    from xatu_amd import capi
    print(f"[sums] {n}x{n}, {natoms} atoms, cutoff {cutoff}", flush=True)
    rng = np.random.default_rng(n)
    a = 2.5
    bravais = a * np.array([[1.0, 0.0, 0.0], [np.cos(np.radians(angle)), np.sin(np.radians(angle)), 0.0]])
    tau = np.concatenate([rng.uniform(0, a, (natoms, 2)), np.zeros((natoms, 1))], axis=1)
    ctx = capi.Context(0)
    ctx.set_lattice(bravais, tau, [1] * natoms, n)
    ctx.fourier_sums(1, 1, 10.0, cutoff, ncell, n * n, regularization=a, potential=capi.XATU_POTENTIAL_COULOMB)
    cells = ctx.get_cells()
    ft, _ = ctx.get_fourier()
    ctx.close()

    c = np.arange(n)
    t = 2 * c - n + (n & 1)
    m = np.arange(ncell) - ncell // 2
    root = np.exp(1j * np.pi * ((t[:, None] * m[None, :]) % (2 * n)) / n)
    R = cells @ bravais
    for i in range(natoms):
        for j in range(i, natoms):
            r = np.linalg.norm(R + tau[i] - tau[j], axis=1)
            v = PREF / np.where(r == 0, a, r) * (r <= a * cutoff + 1e-5)
            table = np.zeros((ncell, ncell))
            table[cells[:, 0] + ncell // 2, cells[:, 1] + ncell // 2] = v
            ref = (root @ (table @ root.T)).T.ravel() / n ** 2  # first coordinate fastest
            bound = (2 * ncell + 16) * 2.0 ** -53 * np.abs(v).sum() / n ** 2
            got = ft[i, j] if i != j else ft[i, i].conj()
            assert np.abs(got - ref).max() <= bound
            assert np.array_equal(ft[j, i], got.conj())
