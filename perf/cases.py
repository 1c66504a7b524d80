"""What the speed of this framework is measured on: calls that a program makes through the C-ABI
binding (``xatu_amd.capi``), over the sizes of the configurations, tests and benchmark of this
repository.

A case is a dict of plain values. ``prepare`` makes what such a program holds before the call (a
context with its lattice and band stacks; for products and gradients also the prepared or resident
operator and the vectors), ``run`` is one call sequence with its results, ``work`` the bytes and
operations it cannot do without, ``exact`` its results from plain torch in 64 bits.

Kinds of calls
  sums       lattice Fourier sums of the screened interaction and their read-back
  solve      lattice sums (or reciprocal-space sums), assembly of the matrix (or preparation of the
             matrix-free operator) and the lowest exciton energies: one point of a scan over
             screening lengths, momenta or models
  gradients  Hellmann-Feynman and band-data gradients of given exciton states
  dense      Y = H X with the resident FP64 matrix on device-resident vectors
  conv       Y = H X matrix-free, on vectors that the program holds on the host

The models are the seeded tight-binding models of ``xatu_amd.synthetic``; another seed gives other
hoppings and onsite energies, hence other bands, band vectors and exciton energies.
"""
import math

import numpy as np
import torch

from xatu_amd import capi, synthetic

# Defaults of a case: the interaction of the benchmark workloads (Keldysh, exchange on).
BASE = dict(natoms=3, orbitals=6, mesh=48, nv=2, nc=2, cutoff=25.0, r0=40.0, eps_m=1.0, eps_s=1.0,
            exchange=True, q=0.0, precision="fp64", matrix_free=False, method="davidson", nstates=16, block=32,
            g_vectors=0, nvec=32, copy_out=False)

# FP64 residual (eV) to which the energies are converged: tight enough that the energies themselves, whose
# error goes with its square, agree to the digits that a comparison of two programs looks at.
TOL = 1e-7


def _case(name, kind, **kw):
    c = dict(BASE, kind=kind, **kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # two-band model on the 20 x 20 mesh of the regression tests: the matrix returned to the
        # caller and every eigenpair ("diag"), the smallest complete calculation
        _case("two_band_20_diag", "solve", natoms=2, orbitals=1, nv=1, nc=1, mesh=20, cutoff=8.0, r0=10.0,
              exchange=False, method="diag", nstates=400, copy_out=True),
        # the same model on the 30 x 30 mesh with 20 cells, lowest 8 with the solver's own block size:
        # launches and latency
        _case("two_band_30_davidson", "solve", natoms=2, orbitals=1, nv=1, nc=1, mesh=30, cutoff=20.0, r0=10.0,
              nstates=8, block=0),
        # unequal band numbers, an odd mesh and a finite momentum: the element-wise assembly and, at an
        # odd dimension, the products on the FP32 matrix cores
        _case("ragged_25_mixed", "solve", mesh=25, nv=1, nc=3, cutoff=10.0, r0=15.0, q=0.05, precision="fp32",
              nstates=4, block=0),
        # the gradient workload: 18 orbitals, 36 x 36, eight states, two screening parameters and the
        # band data (from which the caller forms the hopping gradients)
        _case("gradients_36", "gradients", mesh=36, nstates=8),
        # the 18-orbital model at the middle size, mixed precision
        _case("mixed_48", "solve", mesh=48, precision="fp32"),
        # reciprocal-space interaction (sums over G), FP64, 40 x 40
        _case("reciprocal_40", "solve", mesh=40, cutoff=3.0, g_vectors=5, exchange=False, nstates=8, block=0),
        # the benchmark's default workload, mixed and FP64
        _case("mixed_96", "solve", mesh=96, precision="fp32"),
        _case("fp64_96", "solve", mesh=96),
        # the largest workload: 36 orbitals, 120 x 120, three bands on each side, matrix-free
        _case("matrix_free_120", "solve", natoms=4, orbitals=9, nv=3, nc=3, mesh=120, precision="fp32",
              matrix_free=True),
        # the interaction alone, read back, as a scan over screening lengths uses it
        _case("sums_120", "sums", natoms=4, orbitals=9, mesh=120, q=0.05),
        # a few vectors on the device times the resident matrix: a serving or propagation loop
        _case("dense_36_8", "dense", mesh=36, nvec=8),
        # matrix-free FP64 product for a caller's own iterative solver
        _case("conv_60_16", "conv", mesh=60, nvec=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve_free", "sums", "gradients", "dense", "conv"])
    natoms = rng.randint(2, 4)
    c = dict(natoms=natoms, r0=round(rng.uniform(8.0, 45.0), 2), eps_s=round(rng.uniform(1.0, 4.0), 2),
             exchange=rng.random() < 0.7, q=rng.choice([0.0, 0.0, round(rng.uniform(0.01, 0.2), 3)]))
    if kind == "sums":
        mesh = _log_int(rng, 16, 128)
        return _case(None, kind, **dict(c, orbitals=2, mesh=mesh, cutoff=round(rng.uniform(0.2, 0.5) * mesh, 1)))
    if kind == "gradients":
        nb = rng.randint(1, 2)
        mesh = _log_int(rng, 12, 40)
        return _case(None, kind, **dict(c, orbitals=rng.randint(2 * nb, 8), nv=nb, nc=nb, mesh=mesh,
                                        cutoff=round(0.4 * mesh, 1), nstates=rng.randint(1, 8)))
    nv, nc = rng.choice([(1, 1), (2, 2), (2, 2), (3, 3), (1, 2), (2, 1), (3, 2)])
    orbitals = rng.randint(max(2, -(-2 * max(nv, nc) // natoms)), 9)
    c.update(orbitals=orbitals, nv=nv, nc=nc)
    if kind in ("conv", "solve_free"):
        # FP64 correlations of the mesh, one per pair of orbitals and vector, within the largest listed ones
        mesh = _log_int(rng, 24, 120)
        while (natoms * orbitals * mesh) ** 2 > (36 * 120) ** 2 or nv * nc * mesh ** 2 > 129600:
            mesh -= 1
        c.update(mesh=mesh, cutoff=round(min(30.0, 0.4 * mesh), 1))
        if kind == "conv":
            return _case(None, kind, **dict(c, nvec=rng.randint(1, 32)))
        c["precision"] = rng.choice(["fp64", "fp32", "fp32"])
        if natoms * orbitals > 20 or mesh > 96:
            c["precision"] = "fp32"
        n = rng.randint(2, 16)
        return _case(None, "solve", **dict(c, matrix_free=True, nstates=n, block=2 * n))
    dim = _log_int(rng, 400, 9216 if kind == "dense" or (nv, nc) in ((1, 2), (2, 1), (3, 2)) else 36864)
    mesh = max(12, int(math.sqrt(dim / (nv * nc))))
    c.update(mesh=mesh, cutoff=round(min(30.0, 0.4 * mesh), 1))
    if kind == "dense":
        return _case(None, kind, **dict(c, nvec=rng.randint(1, 32)))
    if rng.random() < 0.2 and mesh <= 60:
        c.update(g_vectors=rng.choice([3, 5, 7]), cutoff=4.0, exchange=False)
    n = rng.randint(2, 16)
    return _case(None, kind, **dict(c, precision=rng.choice(["fp64", "fp32"]), nstates=n, block=rng.choice([0, 2 * n])))


# ---- the model on the mesh ----


def _offsets(n):
    """Integer mesh coordinates of the k-points, first axis fastest."""
    i = np.arange(n * n)
    return np.stack([i % n, i // n], axis=1).astype(np.int32)


def _bands(case, seed):
    """Band stacks of the seeded model: energies nb x nk and vectors norb x nb x nk at k and k + Q, the
    nv bands below and the nc bands above the filling."""
    bravais, motif, cells, H, filling = synthetic.model_arrays(case["natoms"], case["orbitals"], seed=seed)
    n, nv, nc = case["mesh"], case["nv"], case["nc"]
    norb = H.shape[-1]
    filling = min(max(filling, nv), norb - nc)
    recip = 2 * np.pi * np.linalg.inv(bravais[:, :2]).T
    t = (2 * _offsets(n) - n + (n & 1)) / (2.0 * n)

    def stack(shift):
        k = t @ recip + np.array([shift, 0.0])
        phase = torch.from_numpy(np.exp(1j * (k @ cells[:, :2].T)))
        hk = (phase @ torch.from_numpy(H.reshape(len(H), -1))).reshape(n * n, norb, norb)
        w, v = torch.linalg.eigh(hk)
        w, v = w[:, filling - nv:filling + nc], v[:, :, filling - nv:filling + nc]
        # the sum of a vector's coefficients is real and positive
        s = v.sum(1, keepdim=True)
        v = v * (s.conj() / s.abs().clamp_min(1e-300))
        return np.asfortranarray(w.numpy().T), np.asfortranarray(v.permute(1, 2, 0).numpy())

    ek, vk = stack(0.0)
    ekq, vkq = (ek, vk) if case["q"] == 0.0 else stack(case["q"])
    return dict(bravais=bravais, motif=motif[:, :3], recip=recip, ek=ek, vk=vk, ekq=ekq, vkq=vkq)


def _interaction(case):
    kw = dict(eps_m=case["eps_m"], eps_s=case["eps_s"], r0=case["r0"], cutoff=case["cutoff"], ncell=case["mesh"],
              total_cells=case["mesh"] ** 2, exchange=case["exchange"], Q=(case["q"], 0.0, 0.0))
    if case["g_vectors"]:
        kw.update(mode=capi.XATU_MODE_RECIPROCAL, n_reciprocal=case["g_vectors"])
    return kw


def _states(case, seed, count):
    """Normalised exciton-like vectors: envelopes around a k-point times random band weights."""
    rng = np.random.default_rng([seed, 77])
    n, ncv = case["mesh"], case["nv"] * case["nc"]
    off = _offsets(n)
    out = np.empty((n * n, ncv, count), dtype=np.complex128)
    for s in range(count):
        d = (off - rng.integers(0, n, 2) + n // 2) % n - n // 2
        env = np.exp(-(d ** 2).sum(1) / (2.0 * (n * rng.uniform(0.05, 0.25)) ** 2)) + 0.02
        noise = rng.normal(size=(n * n, ncv)) + 1j * rng.normal(size=(n * n, ncv))
        out[:, :, s] = env[:, None] * (noise + rng.normal(size=ncv) + 1j * rng.normal(size=ncv))
    out = out.reshape(n * n * ncv, count)
    return np.asfortranarray(out / np.linalg.norm(out, axis=0))


def prepare(case, seed):
    m = _bands(case, seed) if case["kind"] != "sums" else None
    ctx = capi.Context(0)
    if m is None:
        bravais, motif, _, _, _ = synthetic.model_arrays(case["natoms"], case["orbitals"], seed=seed)
        rng = np.random.default_rng([seed, 5])  # a relaxed motif: the positions differ from seed to seed
        motif = motif[:, :3] + rng.uniform(-0.1, 0.1, (case["natoms"], 3)) * [1.0, 1.0, 0.5]
        ctx.set_lattice(bravais, motif, [case["orbitals"]] * case["natoms"], case["mesh"])
        return dict(case=case, ctx=ctx)
    ctx.set_lattice(m["bravais"], m["motif"], [case["orbitals"]] * case["natoms"], case["mesh"])
    ctx.set_bands(case["nv"], case["nc"], m["ek"], m["vk"], _offsets(case["mesh"]), m["ekq"], m["vkq"])
    s = dict(case=case, ctx=ctx)
    if case["kind"] == "solve":
        return s
    ctx.fourier_sums(**_interaction(case))
    if case["kind"] == "dense":
        ctx.build(capi.XATU_FP64)
        x = torch.from_numpy(np.ascontiguousarray(_states(case, seed, case["nvec"]).T)).cuda()
        s.update(x=x, y=torch.empty_like(x))  # one vector after the other: N x nvec column-major
        torch.cuda.synchronize()
    else:
        ctx.build(capi.XATU_MATRIX_FREE)
        s["x"] = _states(case, seed, case["nvec"] if case["kind"] == "conv" else case["nstates"])
    return s


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    prec = capi.XATU_FP32 if case["precision"] == "fp32" else capi.XATU_FP64
    if kind == "sums":
        ctx.fourier_sums(**_interaction(case))
        ft, ftq = ctx.get_fourier()
        return {"ft": ft, "ftq": ftq}
    if kind == "solve":
        ctx.fourier_sums(**_interaction(case))
        h = ctx.build(capi.XATU_MATRIX_FREE if case["matrix_free"] else prec, copy_out=case["copy_out"])
        diag = case["method"] == "diag"
        w, _, _ = ctx.solve(method=capi.XATU_SOLVE_DIAG if diag else capi.XATU_SOLVE_DAVIDSON, nstates=case["nstates"],
                            precision=prec, matrix_free=case["matrix_free"], block=case["block"], tol=TOL,
                            want_vectors=False)
        return {"energies": w, "matrix": h} if case["copy_out"] else {"energies": w}
    if kind == "gradients":
        hf = ctx.hf_gradients(case["nstates"], [capi.XATU_PARAM_R0, capi.XATU_PARAM_EPS_S], eigvec=state["x"])
        w, g = ctx.band_gradients(case["nstates"], eigvec=state["x"])
        return {"screening": hf, "band_energies": w, "band_vectors": g}
    if kind == "dense":
        ctx.matvec_noalloc(state["x"].data_ptr(), state["y"].data_ptr(), case["nvec"])
        return state["y"]
    return ctx.matvec(state["x"], precision=prec, matrix_free=capi.XATU_MATRIX_FREE_CONV)


def work(case):
    """Each input read and each output written once; operations of the definition evaluated the cheapest
    way the path allows: transforms for sums and convolutions, 8 per complex multiply-add."""
    n, na, nv, nc = case["mesh"], case["natoms"], case["nv"], case["nc"]
    m, norb, ncv = n * n, case["natoms"] * case["orbitals"], nv * nc
    dim = m * ncv
    cells = min(m, int(2 * math.pi / math.sqrt(3) * case["cutoff"] ** 2))
    lg = math.log2(m)
    table = 16.0 * na * na * m
    sums = dict(bytes=table + 8.0 * na * na * cells, flops=2.5 * m * lg * na * (na + 1) + 100.0 * cells * na * na)
    stacks = 2 * 16.0 * norb * (nv + nc) * m

    def product(vectors, real_bytes):
        # matrix-free: the vectors, the band stacks and the table
        return dict(bytes=2 * 16.0 * dim * vectors + stacks + table * real_bytes / 8,
                    flops=vectors * (10.0 * m * lg * norb ** 2 + 8.0 * m * norb ** 2 * 2 * nc + 16.0 * m * norb * ncv))

    kind = case["kind"]
    if kind == "sums":
        return sums
    if kind == "dense":
        return dict(bytes=8.0 * dim * (dim + 1) + 32.0 * dim * case["nvec"], flops=8.0 * dim * dim * case["nvec"])
    if kind == "conv":
        return product(case["nvec"], 8 if case["precision"] == "fp64" else 4)
    if kind == "gradients":
        p = product(case["nstates"], 8)
        return dict(bytes=p["bytes"] + case["nstates"] * stacks, flops=2 * p["flops"])
    if case["method"] == "diag":
        return dict(bytes=sums["bytes"] + stacks + 32.0 * dim * dim, flops=sums["flops"] + 16.0 / 3 * 4 * dim ** 3)
    # about twenty block products and their projections
    block = case["block"] or max(2 * case["nstates"], 8)
    its = 20
    proj = its * 8.0 * dim * 5 * (2.5 * block) * block
    if case["matrix_free"]:
        p = product(block, 4 if case["precision"] == "fp32" else 8)
        return dict(bytes=sums["bytes"] + its * p["bytes"], flops=sums["flops"] + its * p["flops"] + proj)
    size = 4.0 if case["precision"] == "fp32" else 8.0  # half of the Hermitian matrix
    build = 8.0 * dim * dim / 2 * (norb * (nc ** 2 + nv ** 2) / ncv ** 2 + 2 * na * na / ncv + na)
    return dict(bytes=sums["bytes"] + stacks + (1 + its) * size * dim * dim,
                flops=sums["flops"] + build + its * 8.0 * dim * dim * block + proj)


# ---- the same results from plain torch in 64 bits ----


def _cells(case, bravais):
    n = case["mesh"]
    i = np.arange(n * n)
    m = np.stack([i % n, i // n], axis=1) - n // 2
    a = np.linalg.norm(bravais[0])
    return m[np.linalg.norm(m @ bravais, axis=1) < a * case["cutoff"] + 1e-5]


def _struve_minus_y0(x):
    """H0(x) - Y0(x) as the potential is defined: the power series of H0 up to x = 20 and beyond it the
    asymptotic series with the rational approximation of Y0 (Zhang and Jin, STVH0)."""
    x = torch.as_tensor(x, dtype=torch.float64)
    out = torch.empty_like(x)
    lo = x <= 20.0
    xs, s, r = x[lo], torch.ones_like(x[lo]), torch.ones_like(x[lo])
    for k in range(1, 61):
        r = -r * (xs / (2 * k + 1)) ** 2
        s = s + r
    out[lo] = 2 * xs / math.pi * s
    xb = x[~lo]
    km = torch.where(xb >= 50, torch.full_like(xb, 25.0), torch.floor(0.5 * (xb + 1)))
    s, r = torch.ones_like(xb), torch.ones_like(xb)
    live = torch.ones_like(xb, dtype=torch.bool)
    for k in range(1, 26):
        live = live & (k <= km)
        r = torch.where(live, -r * ((2 * k - 1) / xb) ** 2, r)
        s = torch.where(live, s + r, s)
        live = live & (r.abs() >= s.abs() * 1e-12)
    t = 4 / xb
    u = t * t
    p = ((((-.37043e-5 * u + .173565e-4) * u - .487613e-4) * u + .17343e-3) * u - 0.1753062e-2) * u + .3989422793
    q = t * (((((.32312e-5 * u - 0.142078e-4) * u + 0.342468e-4) * u - 0.869791e-4) * u + 0.4564324e-3) * u
             - 0.0124669441)
    th = xb - 0.25 * math.pi
    out[~lo] = 2 / (math.pi * xb) * s + 2 / torch.sqrt(xb) * (p * torch.sin(th) + q * torch.cos(th))
    return out - torch.special.bessel_y0(x)


def _dxf(x):
    """d(x f)/dx for f = H0 - Y0, as (2/pi) int_0^inf e^(-x t) t^2 (1 + t^2)^(-3/2) dt (exp-sinh rule)."""
    x = torch.as_tensor(x, dtype=torch.float64)
    h = 1.0 / 64
    j = torch.arange(-4 * 64, 4 * 64 + 1, dtype=torch.float64) * h
    t = torch.exp(math.pi / 2 * torch.sinh(j))
    w = h * math.pi / 2 * torch.cosh(j) * t * (t * t) * (1 + t * t) ** -1.5
    f = torch.exp(-x[..., None] * t) * w
    return 2 / math.pi * torch.nan_to_num(f).sum(-1)


def _potential(case, bravais, motif, derivative=None):
    """V_ab(R) (natoms x natoms x cells) and, with ``derivative``, its derivative by r0 or eps_s."""
    cells = _cells(case, bravais)
    d = (cells @ bravais)[None, None] + motif[:, None, None] - motif[None, :, None]
    r = torch.from_numpy(np.linalg.norm(d, axis=-1))
    a = float(np.linalg.norm(bravais[0]))
    eps = (case["eps_m"] + case["eps_s"]) / 2
    pref = 1.6021766e-19 / (8e-10 * 8.8541878e-12 * eps * case["r0"])
    x = torch.where(r == 0, torch.full_like(r, a), r) / case["r0"]
    if derivative == "r0":
        v = -pref / case["r0"] * _dxf(x)
    else:
        v = pref * _struve_minus_y0(x.reshape(-1)).reshape(x.shape)
        if derivative == "eps":
            v = -v / (2 * eps)
    return cells, torch.where((r > a * case["cutoff"] + 1e-5), torch.zeros_like(v), v)


def _sums(case, cells, v, recip, bravais):
    """ft[a, b, q] on the mesh and at Q from the table (a < b: the sum; below the conjugate; the diagonal
    holds the conjugate of its sum)."""
    n, na = case["mesh"], case["natoms"]
    t = 2 * _offsets(n).astype(np.int64) - n + (n & 1)
    ph = torch.from_numpy((t @ cells.astype(np.int64).T) % (2 * n))
    root = torch.from_numpy(np.exp(1j * np.pi * np.arange(2 * n) / n)).to(v.device)
    w = root[ph.to(v.device)]
    full = (v.reshape(na * na, -1).to(w.dtype) @ w.T).reshape(na, na, -1) / n ** 2
    q = torch.from_numpy(np.exp(1j * case["q"] * (cells @ bravais)[:, 0])).to(v.device)
    fq = (v.reshape(na * na, -1).to(w.dtype) @ q).reshape(na, na) / n ** 2
    ia, ib = np.triu_indices(na, 1)

    def filled(s):
        o = s.conj().transpose(0, 1).clone()
        o[ia, ib] = s[ia, ib]
        return o

    return filled(full), filled(fq) if case["exchange"] else torch.zeros_like(fq)


def _reciprocal_table(case, m):
    """M_ab(k - k') for every raw difference of mesh points (axis order: difference j, then i)."""
    n, g = case["mesh"], case["g_vectors"]
    i = np.arange(g * g)
    gm = np.stack([i % g, i // g], axis=1) - g // 2
    gv = gm @ m["recip"]
    b1 = np.linalg.norm(m["recip"][0])
    gv = gv[np.linalg.norm(gv, axis=1) < case["cutoff"] * b1 + 1e-5]
    area = abs(np.linalg.det(m["bravais"][:, :2]))
    pref = 1.6021766e-19 * 1e10 / (2 * 8.8541878e-12 * (case["eps_m"] + case["eps_s"]) / 2 * area * n ** 2)
    d = np.arange(-(n - 1), n)
    q = (d[None, :, None] * m["recip"][0] + d[:, None, None] * m["recip"][1]) / n
    tau = m["motif"][:, None, :2] - m["motif"][None, :, :2]
    out = np.zeros((case["natoms"],) * 2 + (2 * n - 1, 2 * n - 1), dtype=np.complex128)
    for v in gv:
        x = q + v
        r = np.linalg.norm(x, axis=-1)
        w = np.where(r < b1 / n ** 2, 0.0, pref / np.maximum(r, 1e-300) / (1 + case["r0"] * r))
        out += w * np.exp(1j * np.einsum("abx,jix->abji", tau, x))
    return torch.from_numpy(out)


def _operator(case, m, dev):
    """(C, V, e, M, MQ) on the device: conduction vectors (k, c, orbital), valence vectors, pair energies
    (k, c, v), the table and its value at Q."""
    nv = case["nv"]
    C = torch.from_numpy(np.ascontiguousarray(m["vkq"][:, nv:].transpose(2, 1, 0))).to(dev)
    V = torch.from_numpy(np.ascontiguousarray(m["vk"][:, :nv].transpose(2, 1, 0))).to(dev)
    e = torch.from_numpy(m["ekq"][nv:].T[:, :, None] - m["ek"][:nv].T[:, None, :]).to(dev)
    if case["g_vectors"]:
        return C, V, e, _reciprocal_table(case, m).to(dev), None
    cells, v = _potential(case, m["bravais"], m["motif"])
    ft, fq = _sums(case, cells, v.to(dev), m["recip"], m["bravais"])
    return C, V, e, ft, fq


def _exchange(case, C, V, MQ):
    """E1, E2 (atom, row) of the exchange term."""
    na, o = case["natoms"], case["orbitals"]
    rho = (C.conj()[:, :, None, :] * V[:, None, :, :]).reshape(-1, na, o).sum(-1).T
    return rho, MQ @ rho.conj()


def _matrix(case, m, dev):
    """The whole BSE matrix."""
    n, na, o = case["mesh"], case["natoms"], case["orbitals"]
    C, V, e, M, MQ = _operator(case, m, dev)
    nk, nc, nv = n * n, case["nc"], case["nv"]
    off = torch.from_numpy(_offsets(n)).to(dev).long()
    H = torch.zeros((nk, nc, nv, nk, nc, nv), dtype=torch.complex128, device=dev)
    if case["g_vectors"]:
        d = off[:, None] - off[None] + n - 1
        at = d[..., 1] * (2 * n - 1) + d[..., 0]
    else:
        d = (off[None] - off[:, None] + n // 2) % n
        at = d[..., 1] * n + d[..., 0]
    M = M.reshape(na, na, -1)
    for b in range(na):
        x = V[:, :, b * o:(b + 1) * o].reshape(nk * nv, o)
        rv = (x @ x.conj().T).reshape(nk, 1, nv, nk, 1, nv)
        t = torch.zeros((nk, nc, nk, nc), dtype=torch.complex128, device=dev)
        for a in range(na):
            y = C[:, :, a * o:(a + 1) * o].reshape(nk * nc, o)
            t += (y.conj() @ y.T).reshape(nk, nc, nk, nc) * M[a, b][at][:, None, :, None]
        H += t[:, :, None, :, :, None] * rv
    H = H.reshape(nk * nc * nv, -1)
    if case["exchange"]:
        e1, e2 = _exchange(case, C, V, MQ)
        H -= e1.T @ e2
    H = -torch.triu(H)
    H += torch.triu(H, 1).mH.contiguous()
    i = torch.arange(len(H), device=dev)
    H[i, i] = (H[i, i].real + e.reshape(-1)).to(H.dtype)
    return H


def _energy(case, C, V, e, M, MQ, psi):
    """psi^H H psi of one state (k, c, v), by transforms: differentiable in every argument."""
    n, na, o = case["mesh"], case["natoms"], case["orbitals"]
    z = torch.matmul(C.transpose(1, 2), psi @ V.conj())  # (k, orbital, orbital)
    z = torch.fft.fft2(z.reshape(n, n, na * o, na * o), dim=(0, 1))
    s = (z.real ** 2 + z.imag ** 2).reshape(n, n, na, o, na, o).sum((3, 5)) / n ** 2
    grid = torch.roll(M.reshape(na, na, n, n), (-(n // 2), -(n // 2)), (2, 3))  # entry of the difference d at d
    p = torch.fft.ifft2(grid, dim=(2, 3)) * n ** 2
    direct = (p.permute(2, 3, 0, 1) * s).sum().real
    x = psi.reshape(-1)
    w = x.real ** 2 + x.imag ** 2
    out = (w * e.reshape(-1)).sum() - direct
    if case["exchange"]:
        e1, e2 = _exchange(case, C, V, MQ)
        f, g = e1 * x.conj(), e2 * x
        before = torch.cumsum(f, 1) - f
        out = out + (2 * (before * g).sum() + (f * g).sum()).real
    return out


def _product(case, C, V, e, M, MQ, X):
    """H X (N x vectors) by transforms."""
    n, na, o = case["mesh"], case["natoms"], case["orbitals"]
    nk, nc, nv = n * n, case["nc"], case["nv"]
    grid = torch.roll(M.reshape(na, na, n, n), (-(n // 2), -(n // 2)), (2, 3))
    p = torch.fft.ifft2(grid, dim=(2, 3)) * n ** 2
    p = p.permute(2, 3, 0, 1)[:, :, :, None, :, None]
    out = []
    for x in X.T:
        psi = x.reshape(nk, nc, nv)
        z = torch.matmul(C.transpose(1, 2), psi @ V.conj())
        z = torch.fft.fft2(z.reshape(n, n, na * o, na * o), dim=(0, 1)).reshape(n, n, na, o, na, o)
        w = torch.fft.ifft2((z * p).reshape(n, n, na * o, na * o), dim=(0, 1)).reshape(nk, na * o, na * o)
        y = e * psi - torch.matmul(torch.matmul(C.conj(), w), V.transpose(1, 2).contiguous())
        y = y.reshape(-1)
        if case["exchange"]:
            e1, e2 = _exchange(case, C, V, MQ)
            a, b = e2 * x, e1.conj() * x
            after = a.sum(1, keepdim=True) - torch.cumsum(a, 1)
            before = torch.cumsum(b, 1) - b
            y = y + (e1 * after + e2.conj() * before).sum(0) + (e1 * e2).sum(0).real * x
        out.append(y)
    return torch.stack(out)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind, n, na = case["kind"], case["mesh"], case["natoms"]
    if kind == "sums":
        bravais, motif, _, _, _ = synthetic.model_arrays(na, case["orbitals"], seed=seed)
        rng = np.random.default_rng([seed, 5])
        motif = motif[:, :3] + rng.uniform(-0.1, 0.1, (na, 3)) * [1.0, 1.0, 0.5]
        cells, v = _potential(case, bravais, motif)
        ft, fq = _sums(case, cells, v.to(dev), None, bravais)
        return {"ft": ft.cpu().numpy(), "ftq": fq.cpu().numpy()}
    dim = n * n * case["nv"] * case["nc"]
    if kind == "solve":
        if dim > 2500:
            return None  # every eigenvalue in 64 bits takes too long
        H = _matrix(case, _bands(case, seed), dev).cpu()
        w = torch.linalg.eigvalsh(H)[:case["nstates"]].numpy()
        return {"energies": w, "matrix": H.numpy()} if case["copy_out"] else {"energies": w}
    m = _bands(case, seed)
    C, V, e, M, MQ = _operator(case, m, dev)
    if kind in ("dense", "conv"):
        x = torch.from_numpy(_states(case, seed, case["nvec"])).to(dev)
        y = _product(case, C, V, e, M, MQ, x).cpu()
        return y if kind == "dense" else y.numpy().T
    # gradients: differentiate the energy by the table, the band energies and the band vectors
    psi = torch.from_numpy(_states(case, seed, case["nstates"])).to(dev)
    cells, v = _potential(case, m["bravais"], m["motif"])
    dv = [_potential(case, m["bravais"], m["motif"], d)[1].to(dev) for d in ("r0", "eps")]
    nv, nc, norb, nk = case["nv"], case["nc"], na * case["orbitals"], n * n
    hf = np.zeros((case["nstates"], 2))
    w = np.zeros((case["nstates"], 2, nk, nv + nc))
    g = np.zeros((case["nstates"], 2, nk, nv + nc, norb), dtype=np.complex128)
    for s in range(case["nstates"]):
        tab, c, b, en = (t.clone().requires_grad_(True) for t in (v.to(dev), C, V, e))
        ft, fq = _sums(case, cells, tab, m["recip"], m["bravais"])
        _energy(case, c, b, en, ft, fq, psi[:, s].reshape(nk, nc, nv)).backward()
        for i, d in enumerate(dv):
            hf[s, i] = float((tab.grad * d).sum())
        w[s, 1, :, nv:] = en.grad.sum(2).cpu().numpy()
        w[s, 0, :, :nv] = -en.grad.sum(1).cpu().numpy()
        g[s, 1, :, nv:] = c.grad.cpu().numpy() / 2
        g[s, 0, :, :nv] = b.grad.cpu().numpy() / 2
    return {"screening": hf, "band_energies": w, "band_vectors": g}
