"""Solutions and systems on both sides of the sizes from which columns come in one
copy with their padding, packed on the device, or column by column: the FP32 values
are the FP64 ones rounded, gaps stay untouched."""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


# columns of 3 kB (41 to a copy of 128 kB, 63 to one of 192), of 41 and of 164
@pytest.mark.parametrize("subdiv,R", [(2, 1), (2, 3), (2, 41), (2, 46), (2, 64), (4, 1), (4, 3), (4, 4), (4, 5), (5, 1),
                                      (5, 2), (5, 5)])
@pytest.mark.parametrize("gap", [0, 3])
def test_solution(subdiv, R, gap):
    m = bem.Mesh().icosphere(subdiv, 0.1).set_bc(0, 1, 0).set_chief(C.ball_points(3, 5, 0.04))
    N = m.num_pnts
    s = bem.Solver(m)
    s.assemble(5.0, bem.PREC_FP32)
    s.set_rhs(bem.RHS_PLANE, C.sphere_points(4, R, 1.0), 1.0)
    s.solve(bem.SOLVE_CGLS, tol=1e-6, maxit=60, refine_tol=1e-6, max_refine=2)
    z = np.full((R, N + gap), 7 + 7j, np.complex128)
    x = np.full((R, N + gap), 7 + 7j, np.complex64)
    for _ in range(2):
        assert bem.lib().bem_solver_get_solution_z(s._h, bem._ptr(z), N + gap) == 0
        assert bem.lib().bem_solver_get_solution(s._h, bem._ptr(x), N + gap) == 0
    assert np.array_equal(x[:, :N], z[:, :N].astype(np.complex64))
    assert np.all(z[:, N:] == 7 + 7j) and np.all(x[:, N:] == 7 + 7j)
    assert np.isfinite(z).all() and len(np.unique(z[:, :N])) > N // 2
    s.close()


# a matrix within one copy, past it, and with gaps
@pytest.mark.parametrize("subdiv,gap", [(0, 0), (1, 0), (1, 5), (2, 0), (2, 5)])
def test_system(subdiv, gap):
    m = bem.Mesh().icosphere(subdiv, 0.1).set_bc(0, 1, 0).set_chief(C.ball_points(3, 5, 0.04))
    M, N = m.num_pnts + 5, m.num_pnts
    s = bem.Solver(m)
    s.assemble(5.0, bem.PREC_FP32)
    A = np.full((N, M + gap), 7 + 7j, np.complex64)
    assert bem.lib().bem_solver_get_system(s._h, bem._ptr(A), M + gap, None, 0) == 0
    assert np.array_equal(A[:, :M].T, s.rows(np.arange(M)).astype(np.complex64))
    assert np.all(A[:, M:] == 7 + 7j)
    s.close()
