"""Solves with a factored system by groups of four panels (128 columns), on sizes
around a panel, a group and the rows of a workgroup, against numpy and against
the solve one panel and one column at a time (BEM_QR_PER_COLUMN_SOLVE).

Tolerances: the least-squares solution of a system with condition number c and
relative residual r is off by at most about sqrt(M) u (c + c^2 r), factor 4,
u = 6e-8 (FP32) or 1.1e-16 (FP64).
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


def _tolerance(A, B, X, u):
    sv = np.linalg.svd(A, compute_uv=False)
    c = sv[0] / sv[-1]
    res = np.linalg.norm(B - A @ X) / (sv[0] * np.linalg.norm(X))
    return 4 * np.sqrt(A.shape[0]) * u * (c + c * c * res)


def _lstsq(A, B):
    """numpy's solution with one step of refinement (its own is off by up to
    5e-15, with A^H (B - A X) 30 times that of the solutions tested here)."""
    X = np.linalg.lstsq(A, B, rcond=None)[0]
    return X + np.linalg.lstsq(A, B - A @ X, rcond=None)[0]


@pytest.mark.parametrize("M,N,R", [(1, 1, 1), (63, 31, 2), (65, 33, 1), (96, 96, 3), (128, 97, 1), (127, 127, 1),
                                   (128, 128, 2), (130, 129, 1), (192, 160, 17), (256, 256, 1), (300, 257, 1),
                                   (513, 512, 1), (4160, 130, 2), (4097, 300, 1)])
def test_group_solve_fp32(monkeypatch, M, N, R):
    rng = np.random.default_rng(M + 5 * N)
    A = (rng.standard_normal((M, N)) + 1j * rng.standard_normal((M, N))) / np.sqrt(2 * M)
    A[:N] += 1.5 * np.eye(N)
    A, B = A.astype(np.complex64), (rng.standard_normal((M, R)) + 1j * rng.standard_normal((M, R))).astype(np.complex64)
    X = bem.qr_solve(A, B)
    A64, B64 = A.astype(np.complex128), B.astype(np.complex128)
    X64 = _lstsq(A64, B64)
    tol = _tolerance(A64, B64, X64, 6e-8)
    monkeypatch.setenv("BEM_QR_PER_COLUMN_SOLVE", "1")
    Xc = bem.qr_solve(A, B)
    err = [np.linalg.norm(Y - X64) / np.linalg.norm(X64) for Y in (X, Xc)]
    print("case: %d x %d, %d: groups %.2g, per column %.2g, tolerance %.2g" % (M, N, R, *err, tol), flush=True)
    assert err[0] <= tol and np.linalg.norm(X - Xc) <= tol * np.linalg.norm(X64)


@pytest.mark.parametrize("subdiv,nchief,R", [(0, 0, 1), (1, 3, 2), (2, 0, 1), (2, 30, 3), (3, 8, 1)])
def test_group_solve_fp64(subdiv, nchief, R):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=4, lmax=4, amp=0.03, seed=30 + subdiv)
    m.set_bc(0, 1, 0)
    if nchief:
        m.set_chief(C.ball_points(5, nchief, 0.03))
    k = 14.0
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP64)
    dirs = C.sphere_points(60 + R, R, 1.0)
    s.set_rhs(bem.RHS_PLANE, dirs, 1.0)
    s.solve(bem.SOLVE_QR)
    X = s.solution()
    A = s.rows(np.arange(m.num_pnts + nchief))
    s.close()
    x = np.vstack([m.pnts(), m.chief().reshape(-1, 3)]).astype(np.float64)
    B = np.exp(-1j * k * x @ dirs.astype(np.float64).T)
    X0 = _lstsq(A, B)
    # (the right-hand sides are formed with a phase rounded to 1.2e-16 k |x|)
    tol = _tolerance(A, B, X0, 1.1e-16)
    assert np.linalg.norm(X - X0) <= tol * np.linalg.norm(X0)
