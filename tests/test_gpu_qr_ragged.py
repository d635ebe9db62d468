"""QR least squares whose last panel is narrow (N no multiple of 32), on heights
around the panel kernels' limits, against numpy's FP64 least squares.

Tolerance: Householder QR in FP32 is backward stable; the solution of a well
conditioned system (condition number c) is off by at most about
sqrt(M) * 6e-8 * c, with a factor 4 for the constants.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem

pytestmark = pytest.mark.gpu


def system(rng, M, N, R):
    A = (rng.standard_normal((M, N)) + 1j * rng.standard_normal((M, N))) / np.sqrt(2 * M)
    A[:N] += 1.5 * np.eye(N)  # like a collocation matrix: a dominant diagonal
    B = rng.standard_normal((M, R)) + 1j * rng.standard_normal((M, R))
    return A.astype(np.complex64), B.astype(np.complex64)


@pytest.mark.parametrize("M,N,R", [(1, 1, 1), (3, 2, 2), (33, 31, 1), (34, 33, 3), (164, 162, 3), (257, 250, 1),
                                   (520, 513, 2), (1025, 1022, 1), (1100, 1057, 17), (2050, 1095, 1)])
def test_qr_ragged_sizes(M, N, R):
    rng = np.random.default_rng(M * 7 + N)
    A, B = system(rng, M, N, R)
    X = bem.qr_solve(A, B)
    A64, B64 = A.astype(np.complex128), B.astype(np.complex128)
    X64 = np.linalg.lstsq(A64, B64, rcond=None)[0]
    sv = np.linalg.svd(A64, compute_uv=False)
    # an inconsistent system: the residual enters with the condition number squared
    c = sv[0] / sv[-1]
    res = np.linalg.norm(B64 - A64 @ X64) / (sv[0] * np.linalg.norm(X64))
    tol = 4 * np.sqrt(M) * 6e-8 * (c + c * c * res)
    assert np.all(np.isfinite(X))
    assert np.linalg.norm(X - X64) <= tol * np.linalg.norm(X64)
