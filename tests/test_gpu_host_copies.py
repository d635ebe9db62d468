"""Matrices between the caller's buffers and the device: contiguous columns go
packed, columns with gaps pitched and with the gaps left alone; C- and
Fortran-ordered inputs of the binding give the same results."""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


# 162 + 30 = 192 rows: no padding on the device; 162 and 163: padding
@pytest.mark.parametrize("nchief", [0, 1, 30])
@pytest.mark.parametrize("gap", [0, 5])
def test_system_columns(nchief, gap):
    m = bem.Mesh().icosphere(2, 0.1)
    if nchief:
        m.set_chief(C.ball_points(3, nchief, 0.04))
    M, N = m.num_pnts + nchief, m.num_pnts
    ld = M + gap
    src = np.array([[0.3, 0.1, -0.2], [1e6, 1e6, 1e6]], np.float32)
    A = np.full((N, ld), 7 + 7j, np.complex64)
    B = np.full((2, ld), 7 + 7j, np.complex64)
    assert bem.lib().bem_system(m.handle, 5.0, bem._ptr(src), 2, bem._ptr(A), ld, bem._ptr(B), ld) == 0
    A0, B0 = bem.bem_system(m, 5.0, src)
    assert np.array_equal(A[:, :M].T, A0) and np.array_equal(B[:, :M].T, B0)
    assert np.all(A[:, M:] == 7 + 7j) and np.all(B[:, M:] == 7 + 7j)
    s = bem.Solver(m)
    s.assemble(5.0, bem.PREC_FP32)
    assert np.array_equal(s.rows([0, N // 2, M - 1]).astype(np.complex64), A0[[0, N // 2, M - 1]])
    s.set_rhs(bem.RHS_PLANE, [[0, 0, 1], [1, 0, 0], [0, 1, 0]], 1.0)
    s.solve(bem.SOLVE_QR)
    z = s.solution()
    x = np.full((3, N + gap), 7 + 7j, np.complex64)
    assert bem.lib().bem_solver_get_solution(s._h, bem._ptr(x), N + gap) == 0
    assert np.array_equal(x[:, :N].T, z.astype(np.complex64)) and np.all(x[:, N:] == 7 + 7j)
    zg = np.full((3, N + gap), 7 + 7j, np.complex128)
    assert bem.lib().bem_solver_get_solution_z(s._h, bem._ptr(zg), N + gap) == 0
    assert np.array_equal(zg[:, :N].T, z) and np.all(zg[:, N:] == 7 + 7j)
    s.close()


def test_matrix_orders():
    rng = np.random.default_rng(5)
    A = (rng.standard_normal((70, 65)) + 1j * rng.standard_normal((70, 65)) + 9 * np.eye(70, 65)).astype(np.complex64)
    b = (rng.standard_normal(70) + 1j * rng.standard_normal(70)).astype(np.complex64)
    F, wide = np.asfortranarray(A), np.zeros((140, 130), np.complex64)
    wide[::2, ::2] = A
    keep = F.copy()
    x = bem.qr_solve(A, b)
    for other in (F, wide[::2, ::2], A.astype(np.complex128)):
        assert np.array_equal(bem.qr_solve(other, b), x)
    assert np.array_equal(F, keep)
    X, R, _ = bem.lsq_solve(F, b)
    assert np.array_equal(F, keep) and np.array_equal(bem.lsq_solve(A, b)[1], R)
    y = bem.gmres(A[:65], b[:65], 65, 1e-6)
    assert np.array_equal(bem.gmres(np.asfortranarray(A[:65]), b[:65], 65, 1e-6), y)
