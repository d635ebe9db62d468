"""FP64 QR solves on both sides of 256 unknowns, up to which one workgroup solves a
right-hand side, against numpy's least squares.

Tolerance: the least-squares solution of a system with condition number c and
relative residual r is off by at most about sqrt(M) u (c + c^2 r), factor 4,
u = 1.1e-16; numpy's own is refined once.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C
from test_gpu_block_policy import _sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rings,cols,nchief,R", [(2, 3, 0, 1), (5, 6, 5, 3), (9, 10, 5, 17), (10, 25, 0, 2), (6, 42, 2, 64),
                                                 (14, 18, 30, 3), (15, 17, 3, 3), (17, 15, 0, 64)])
def test_solution(rings, cols, nchief, R):
    p, e = _sphere(rings, cols)
    m = bem.Mesh().set(p, e, (0, 1, 0))
    if nchief:
        m.set_chief(C.ball_points(5, nchief, 0.04))
    k = 14.0
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP64)
    dirs = C.sphere_points(60 + R, R, 1.0)
    s.set_rhs(bem.RHS_PLANE, dirs, 1.0)
    s.solve(bem.SOLVE_QR)
    X = s.solution()
    A = s.rows(np.arange(len(p) + nchief))
    s.close()
    x = np.vstack([p, m.chief().reshape(-1, 3)]).astype(np.float64)
    B = np.exp(-1j * k * x @ dirs.astype(np.float64).T)
    X0 = np.linalg.lstsq(A, B, rcond=None)[0]
    X0 = X0 + np.linalg.lstsq(A, B - A @ X0, rcond=None)[0]
    sv = np.linalg.svd(A, compute_uv=False)
    c = sv[0] / sv[-1]
    res = np.linalg.norm(B - A @ X0) / (sv[0] * np.linalg.norm(X0))
    tol = 4 * np.sqrt(len(x)) * 1.1e-16 * (c + c * c * res)
    err = np.linalg.norm(X - X0) / np.linalg.norm(X0)
    print("case: %d unknowns: error %.2g, tolerance %.2g" % (len(p), err, tol), flush=True)
    assert err <= tol
