"""The Arnoldi step in a product and two launches (the product's partials summed
by the dot kernel, the newest basis vector normalised by the step after it)
against the step with every launch of its own (BEM_ARNOLDI_UNFUSED), on the same
system.

Both run to the same FP64 residual, so a wrong basis shows in the number of
steps, not in the solution: it may differ by the rounding of the last step of
each cycle only.  The solutions differ by at most the two residuals times the
condition number (a few hundred, squared where there are CHIEF rows), 1e-10:
1e-7 and 1e-5.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


def _solve(m, k, prec, R, restart, scale):
    s = bem.Solver(m)
    s.assemble(k, prec)
    s.set_rhs(bem.RHS_PLANE, C.sphere_points(7 + R, R, 1.0), scale)
    st = s.solve(bem.SOLVE_GMRES, restart=restart, tol=1e-6, maxit=4000, refine_tol=1e-10, max_refine=50)
    X = s.solution()
    s.close()
    return X, st


# fewer nodes than a wave, a workgroup's rows, and 512 rows a workgroup; more
# than one group of 16 basis vectors; restarts within a chunk of steps; two
# Gram-Schmidt passes; one matrix of each precision; right-hand sides far from 1
@pytest.mark.parametrize("subdiv,nchief,R,restart,prec,env,scale", [
    (0, 0, 2, 30, 32, None, 1.0), (0, 3, 5, 3, 32, None, 1.0), (1, 0, 1, 30, 32, None, 1.0),
    (2, 0, 16, 7, 32, None, 1e-9), (2, 5, 17, 60, 32, None, 1.0), (3, 0, 33, 60, 32, None, 1e12),
    (3, 9, 2, 60, 32, "BEM_CGS2", 1.0), (3, 9, 1, 40, 32, None, 1.0), (3, 0, 3, 40, 64, None, 1.0),
    (2, 4, 2, 40, 64, "BEM_CGS2", 1.0), (5, 0, 2, 40, 32, None, 1.0)])
def test_arnoldi_step_matches_separate_launches(monkeypatch, subdiv, nchief, R, restart, prec, env, scale):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=4, lmax=4, amp=0.03, seed=90 + subdiv)
    m.set_bc(0, 1, 0)
    if nchief:
        m.set_chief(C.ball_points(8, nchief, 0.03))
    k = 22.0
    prec = bem.PREC_FP64 if prec == 64 else bem.PREC_FP32
    if env:
        monkeypatch.setenv(env, "1")
    X, st = _solve(m, k, prec, R, restart, scale)
    monkeypatch.setenv("BEM_ARNOLDI_UNFUSED", "1")
    X0, st0 = _solve(m, k, prec, R, restart, scale)
    print("case:", st, st0, flush=True)
    assert st["converged"] == 1 and st0["converged"] == 1
    assert abs(st["iterations"] - st0["iterations"]) <= 1 + st0["refinements"]
    err = np.linalg.norm(X - X0, axis=0) / np.linalg.norm(X0, axis=0)
    assert err.max() <= (1e-5 if nchief else 1e-7)
