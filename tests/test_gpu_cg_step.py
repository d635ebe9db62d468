"""The lockstep CG on the normal equations (norms, updates and the sums of the
products' partials in three launches a step) against numpy's least squares on
the same matrix.

The solve ends at |A^H r| <= 1e-11 |A^H b|; with condition numbers of a few
hundred, squared by the normal equations, the solutions agree to 1e-6.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


def _problem(subdiv, nchief, R):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=4, lmax=4, amp=0.03, seed=40 + subdiv)
    m.set_bc(0, 1, 0)
    if nchief:
        m.set_chief(C.ball_points(11, nchief, 0.03))
    k = 16.0
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP32)
    dirs = C.sphere_points(50 + R, R, 1.0)
    s.set_rhs(bem.RHS_PLANE, dirs, 1.0)
    return m, k, s, dirs


# fewer rows than a wave, a workgroup of 256 rows and a few over, several; the
# GEMV (one system), the 16- and the 32-wide products, and one system more
@pytest.mark.parametrize("subdiv,nchief", [(0, 0), (1, 3), (2, 62), (2, 94), (2, 95), (3, 9)])
@pytest.mark.parametrize("R", [1, 2, 16, 17, 33])
def test_cg_matches_least_squares(subdiv, nchief, R):
    m, k, s, dirs = _problem(subdiv, nchief, R)
    st = s.solve(bem.SOLVE_CGLS, tol=1e-6, maxit=6000, refine_tol=1e-11, max_refine=50)
    X = s.solution()
    A = s.rows(np.arange(m.num_pnts + nchief))
    s.close()
    x = np.vstack([m.pnts(), m.chief().reshape(-1, 3)]).astype(np.float64)
    B = np.exp(-1j * k * x @ dirs.astype(np.float64).T)
    X0 = np.linalg.lstsq(A, B, rcond=None)[0]
    err = np.linalg.norm(X - X0, axis=0) / np.linalg.norm(X0, axis=0)
    print("case:", st, err.max(), flush=True)
    assert st["converged"] == 1
    assert err.max() <= 1e-6


# a limit on the steps that is no multiple of a chunk of 8, nor even
@pytest.mark.parametrize("maxit", [1, 7, 8, 13])
def test_cg_stops_at_the_limit(maxit):
    m, k, s, dirs = _problem(2, 5, 3)
    st = s.solve(bem.SOLVE_CGLS, tol=1e-6, maxit=maxit, refine_tol=1e-14, max_refine=50)
    X = s.solution()
    s.close()
    assert st["iterations"] == maxit and np.isfinite(X).all()


# more than 1.2e8 of M N nrhs and 1.5e7 of M N at 16 or fewer right-hand sides: the
# block iteration, whose steps are fewer; one system less: the lockstep one
@pytest.mark.parametrize("R,block", [(1, False), (2, True)])
def test_block_size_policy_few_right_hand_sides(R, block):
    m, k, s, dirs = _problem(5, 16, R)
    st = s.solve(bem.SOLVE_BLOCK_CG, tol=1e-6, maxit=6000, refine_tol=1e-10, max_refine=50)
    X = s.solution()
    sl = s.solve(bem.SOLVE_CGLS, tol=1e-6, maxit=6000, refine_tol=1e-10, max_refine=50)
    Xl = s.solution()
    s.close()
    print("case:", st, sl, flush=True)
    assert st["converged"] == 1 and sl["converged"] == 1
    assert (st["iterations"] < sl["iterations"]) == block
    assert block or np.array_equal(X, Xl)
    # both to 1e-10 on the normal equations (condition numbers as above)
    assert np.linalg.norm(X - Xl) <= 1e-5 * np.linalg.norm(Xl)
