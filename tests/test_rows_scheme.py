"""The scheme of the convolution on row and column transforms (fft_stages.hpp, conv_rows.hpp), restated with the
same index maps and checked on the CPU: the factor pairs and constants as they stand in the source, the two steps of
a side's transform, and the whole correlation with the potential as its spectrum on a window of the first axis."""
import re

import numpy as np
import pytest
from conftest import ROOT

DEVICE = ROOT / "xatu_amd" / "csrc" / "device"
SOURCE = (DEVICE / "fft_stages.hpp").read_text()
LENGTHS = set(range(1, 18)) | {19, 23, 29, 31, 37, 41}
PAIRS = [(int(a), int(b)) for a, b in re.findall(r"X\((\d+), (\d+)\)", SOURCE)]


def test_pairs():
    sides = [a * b for a, b in PAIRS]
    assert len(sides) == len(set(sides)) == 100 and min(sides) == 1 and max(sides) <= 128
    for a, b in PAIRS:
        assert a <= b and a in LENGTHS and b in LENGTHS
        assert b <= 31 or a == 1
    # what is left out: 125 and the sides with a longer prime factor
    for n in range(2, 129):
        p = max(q for q in range(2, n + 1) if n % q == 0 and all(q % d for d in range(2, q)))
        assert (n in sides) == (n != 125 and (p <= 31 or n in (37, 41))), n


def test_constants():
    for length, body in re.findall(r"struct PrimeRoots<(\d+)> \{(.*?)\n\};", SOURCE, re.S):
        p = int(length)
        c, s = (np.array([float(x) for x in re.findall(r"-?\d\.\d+", part)]) for part in body.split("double s["))
        k = np.arange(1, (p - 1) // 2 + 1)
        assert np.abs(c - np.cos(2 * np.pi * k / p)).max() < 1e-15 and np.abs(s - np.sin(2 * np.pi * k / p)).max() < 1e-15
    angles = re.findall(r"case (\d+): return (\d\.\d+);", SOURCE)
    assert len(angles) > 20
    for a, value in angles:
        assert abs(float(value) - np.cos(2 * np.pi * int(a) / 720)) < 1e-15


def dft(v, sign, axis=0):
    n = v.shape[axis]
    k = np.arange(n)
    return np.moveaxis(np.tensordot(np.exp(sign * 2j * np.pi * np.outer(k, k) / n), np.moveaxis(v, axis, 0), 1), 0, axis)


def forward(x, A, B):
    """x[B j2 + s] -> A-point transforms over j2, twiddles, B-point transforms over s, X[k1 + A k2]."""
    n = A * B
    z = dft(x.reshape(A, B), -1, 0)  # k1, s
    z = z * np.exp(-2j * np.pi * np.outer(np.arange(A), np.arange(B)) / n)
    z = dft(z, -1, 1)  # k1, k2
    return z.T.reshape(n)


def inverse(X, A, B):
    """The steps of forward() undone: B-point transforms over k2, conjugated twiddles, A-point transforms over k1."""
    n = A * B
    z = dft(X.reshape(B, A).T, 1, 1)  # k1, s
    z = z * np.exp(2j * np.pi * np.outer(np.arange(A), np.arange(B)) / n)
    return dft(z, 1, 0).reshape(n)


@pytest.mark.parametrize("A,B", PAIRS)
def test_two_steps(A, B):
    n = A * B
    rng = np.random.default_rng(n)
    x = rng.normal(size=n) + 1j * rng.normal(size=n)
    X = forward(x, A, B)
    assert np.abs(X - np.fft.fft(x)).max() < 1e-12 * n
    assert np.abs(inverse(X, A, B) / n - x).max() < 1e-13 * n


@pytest.mark.parametrize("n,reach", [(2, 0), (5, 1), (6, 2), (12, 3), (7, 3), (9, 6), (10, 9), (15, 4)])
@pytest.mark.parametrize("pair", ["a < b", "a >= b"])
def test_correlation(n, reach, pair):
    """w(k) = sum_k' M(k' - k) z(k') with M(Delta) = (1/T) sum_R V(R) e^{i Delta R} (conjugated for a >= b), for
    cells within the window, as wide as the mesh and wider than it (aliases add); holes are zeros of z."""
    rng = np.random.default_rng(n + reach)
    A, B = next(p for p in PAIRS if p[0] * p[1] == n)
    cells = [(m0, m1) for m0 in range(-reach, reach + 1) for m1 in range(-reach - 1, reach + 2)]
    V = rng.normal(size=len(cells))
    total = 3.0 * n
    z = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))  # [o1, o0]
    z[rng.random((n, n)) < 0.2] = 0.0
    # the sum over pairs
    sign = 1 if pair == "a < b" else -1
    w = np.zeros((n, n), complex)
    o = np.arange(n)
    for (m0, m1), v in zip(cells, V):
        e0, e1 = np.exp(sign * 2j * np.pi * m0 * o / n), np.exp(sign * 2j * np.pi * m1 * o / n)
        w += v / total * np.outer(e1.conj(), e0.conj()) * (e1 @ z @ e0)
    # window and spectrum
    W = min(n, 2 * reach + 1)
    w0 = 0 if W == n else n - reach
    P = np.zeros((n, W))  # xi_1, j
    for (m0, m1), v in zip(cells, V):
        x0, x1 = (-sign * m0) % n, (-sign * m1) % n
        P[x1, (x0 - w0) % n] += v / total
    # rows, columns with the spectrum, rows
    G = np.zeros((n, W), complex)
    for o1 in range(n):
        X = forward(z[o1], A, B)
        for xi in range(n):
            j = xi - w0 + (n if xi < w0 else 0)
            if j < W:
                G[o1, j] = X[xi]
    for j in range(W):
        G[:, j] = inverse(forward(G[:, j], A, B) * P[:, j], A, B)
    got = np.zeros((n, n), complex)
    for o1 in range(n):
        X = np.zeros(n, complex)
        for xi in range(n):
            j = xi - w0 + (n if xi < w0 else 0)
            if j < W:
                X[xi] = G[o1, j]
        got[o1] = inverse(X, A, B)
    assert np.abs(got - w).max() < 1e-12 * np.abs(w).max()
