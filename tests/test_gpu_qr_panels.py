"""FP32 QR panels formed from their Gram matrix, with the column-wise algorithm
for the panels that this cannot take, on heights and widths around the kernels'
limits: Q unitary, Q R = A, and R as the column-wise algorithm on every panel
(BEM_QR_GPANEL) gives it.

Tolerances: a panel's reflectors, and its update of each later entry, are off by
at most about 8 roundings (6e-8) of the column's norm, and an entry of the last
column meets N / 32 panels: (8 + N / 4) 6e-8.  R depends on A with the condition
number.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem

pytestmark = pytest.mark.gpu

EPS = 6e-8


def _random(rng, M, N):
    return (rng.standard_normal((M, N)) + 1j * rng.standard_normal((M, N))).astype(np.complex64)


def _check(A, monkeypatch, same_r=True):
    M, N = A.shape
    B = np.ones((M, 1), np.complex64)
    X, R, Q = bem.lsq_solve(A, B, want_q=True)
    monkeypatch.setenv("BEM_QR_GPANEL", "1")
    Xg, Rg, _ = bem.lsq_solve(A, B, want_q=True)
    A64, Q64, R64 = A.astype(np.complex128), Q.astype(np.complex128), np.triu(R[:N].astype(np.complex128))
    tol = (8 + N / 4) * EPS
    unit = np.linalg.norm(Q64.conj().T @ Q64 - np.eye(M)) / np.sqrt(M)
    rec = np.linalg.norm(Q64[:, :N] @ R64 - A64) / max(np.linalg.norm(A64), 1e-300)
    print("case: %d x %d: unitary %.2g, Q R - A %.2g, tolerance %.2g" % (M, N, unit, rec, tol), flush=True)
    assert unit <= tol and rec <= tol
    if same_r:
        c = np.linalg.cond(A64)
        assert np.linalg.norm(R64 - np.triu(Rg[:N])) <= 2 * tol * c * np.linalg.norm(A64)
    return X, R, Xg, Rg


@pytest.mark.parametrize("M,N", [(2, 1), (3, 2), (32, 31), (33, 32), (34, 33), (64, 40), (65, 64),
                                 (97, 96), (200, 7), (1024, 32), (1025, 33), (1100, 100), (2049, 64)])
def test_panels_give_the_factorisation(monkeypatch, M, N):
    _check(_random(np.random.default_rng(M + 3 * N), M, N), monkeypatch)


# square systems (the last column has nothing below its diagonal), solved
@pytest.mark.parametrize("N", [1, 2, 31, 32, 33, 64, 95])
def test_panels_of_square_systems(N):
    rng = np.random.default_rng(N)
    A = _random(rng, N, N) + 2 * np.sqrt(N) * np.eye(N, dtype=np.complex64)
    B = _random(rng, N, 2)
    X = bem.qr_solve(A, B)
    X64 = np.linalg.solve(A.astype(np.complex128), B.astype(np.complex128))
    tol = 2 * (8 + N / 4) * EPS * np.linalg.cond(A.astype(np.complex128))
    assert np.linalg.norm(X - X64) <= tol * np.linalg.norm(X64)


# scales of FP32, and condition numbers of a panel on both sides of the limit
# (3e4) of the Gram matrix
@pytest.mark.parametrize("scale,cond", [(1e-12, 1.0), (1e12, 1.0), (1.0, 1e2), (1.0, 1e4), (1.0, 1e5), (1.0, 1e7)])
def test_panels_scales_and_conditions(monkeypatch, scale, cond):
    rng = np.random.default_rng(9)
    A = _random(rng, 150, 70)
    A[:, 33:60] = A[:, 32:33] + A[:, 33:60] / np.float32(cond)  # close columns in the second panel
    _check((A * np.float32(scale)).astype(np.complex64), monkeypatch, same_r=cond < 1e5)


# columns that are equal, zero, or need no reflection
@pytest.mark.parametrize("kind", ["equal", "zero", "identity", "real", "triangular"])
def test_panels_that_are_not_regular(monkeypatch, kind):
    rng = np.random.default_rng(10)
    A = _random(rng, 130, 50)
    if kind == "equal":
        A[:, 40] = A[:, 35]
    elif kind == "zero":
        A[:, 5] = 0
    elif kind == "identity":
        A = np.eye(130, 50, dtype=np.complex64)
    elif kind == "real":
        A = A.real.astype(np.complex64)
    else:
        A = np.triu(A.real + 9 * np.eye(130, 50)).astype(np.complex64)
    _, R, _, Rg = _check(A, monkeypatch, same_r=kind in ("real", "triangular"))
    if kind in ("identity", "triangular"):  # no reflection: R is A, signs included
        assert np.linalg.norm(R[:50] - A[:50]) <= 1e-6 * np.linalg.norm(A)
        assert np.linalg.norm(R[:50] - Rg[:50]) <= 1e-6 * np.linalg.norm(A)
