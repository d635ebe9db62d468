"""FP32 QR of matrices whose panels the Gram matrix does not take, of which the
later ones go column by column in launches of their own: Q unitary and Q R = A
whatever the order of such panels, and a time within reach of a regular matrix's.

Tolerances: as for panels of either kind, (8 + N / 4) 6e-8.
"""
import time

import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem

pytestmark = pytest.mark.gpu

EPS = 6e-8


def _matrix(M, N, panels, kind):
    rng = np.random.default_rng(M + N)
    A = (rng.standard_normal((M, N)) + 1j * rng.standard_normal((M, N))).astype(np.complex64)
    for p in panels:
        c = A[:, 32 * p:32 * p + 32]
        if kind == "equal":
            c[:, 7] = c[:, 3]
        elif kind == "zero":
            c[:, 5] = 0
        else:  # columns 1e-5 apart
            c[:, 1:] = c[:, :1] + c[:, 1:] * np.float32(1e-5)
    return A


# every panel, the first ones, one in the middle, every other one, the last ones with
# a narrow panel behind; one workgroup of rows, several, more than a wave's tail
@pytest.mark.parametrize("M,N,panels", [(420, 416, range(13)), (700, 400, range(5)), (1100, 400, [6]),
                                        (515, 416, range(0, 13, 2)), (430, 427, [3, 4, 11, 12]), (33, 32, [0]),
                                        (97, 96, [0, 1, 2])])
@pytest.mark.parametrize("kind", ["equal", "zero", "close"])
def test_factorisation(M, N, panels, kind):
    A = _matrix(M, N, panels, kind)
    X, R, Q = bem.lsq_solve(A, np.ones((M, 1), np.complex64), want_q=True)
    A64, Q64, R64 = A.astype(np.complex128), Q.astype(np.complex128), np.triu(R[:N].astype(np.complex128))
    tol = (8 + N / 4) * EPS
    unit = np.linalg.norm(Q64.conj().T @ Q64 - np.eye(M)) / np.sqrt(M)
    rec = np.linalg.norm(Q64[:, :N] @ R64 - A64) / np.linalg.norm(A64)
    print("case: %d x %d: unitary %.2g, Q R - A %.2g, tolerance %.2g" % (M, N, unit, rec, tol), flush=True)
    assert unit <= tol and rec <= tol
    assert np.array_equal(bem.lsq_solve(A, np.ones((M, 1), np.complex64))[1], R)  # the same route each time


# 10300 rows: a panel in one workgroup takes 5.7 ms, in launches by column 0.3; all
# 41 panels that way took 20 times a regular matrix's time
def test_time_without_a_regular_panel():
    def best(A):
        b, t = np.ones(A.shape[0], np.complex64), []
        for _ in range(3):
            t0 = time.perf_counter()
            bem.qr_solve(A, b)
            t.append(time.perf_counter() - t0)
        return min(t)

    M, N = 10300, 41 * 32
    t = [best(np.asfortranarray(_matrix(M, N, panels, "close"))) for panels in ((), range(41))]
    print("case: %.1f ms, %.1f ms" % (1e3 * t[0], 1e3 * t[1]), flush=True)
    assert t[1] <= 8 * t[0]
