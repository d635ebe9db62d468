"""The FP64 path with several right-hand sides (products of up to 8 per pass over
the matrix, groups past that) and its fast assembly, against the oracle.

Matrix tolerance: a dozen FP64 roundings per entry and a phase k r rounded to
1.2e-16 k r, with a factor 10: 1e-14 + 1e-15 k D.  Solutions: refined to a
residual of 1e-12 on the (normal) equations of a matrix with condition numbers
of a few hundred at most, squared where there are CHIEF rows: 1e-8 and 1e-10.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C
import oracle_py as orc

pytestmark = pytest.mark.gpu

AIR = dict(dens=float(np.float32(1.2041)), speed=float(np.float32(343.21)))


@pytest.fixture(autouse=True)
def quadrature():
    orc.quad_init(6)


# element sizes on both sides of the limit up to which an element's phases need
# no quadrant (k rho = 0.79), and far past it
@pytest.mark.parametrize("bc", [(0, 1, 0), (0, 1, -1), (0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j)],
                         ids=["rigid", "source", "impedance"])
@pytest.mark.parametrize("subdiv,kappa,nchief", [(1, 0.3, 0), (2, 0.78, 3), (2, 0.81, 62), (3, 0.05, 8), (2, 5.0, 1),
                                                 (1, 2000.0, 2)])
def test_fp64_assembly_matches_oracle(subdiv, kappa, nchief, bc):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=8, lmax=6, amp=0.05, seed=60 + subdiv)
    m.set_bc(*bc)
    chief = C.ball_points(78, nchief, 0.03) if nchief else np.zeros((0, 3), np.float32)
    if nchief:
        m.set_chief(chief)
    p, e, bcs = C.mesh_arrays(m)
    rho = np.median(np.linalg.norm(p[e] - p[e].mean(1)[:, None], axis=2).max(1))
    k = float(np.float32(kappa / rho))
    A0, _ = orc.assemble(k, np.vstack([p, chief]).astype(np.float64), p.shape[0], e, bcs, dtype=np.float64, **AIR)
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP64)
    A = s.rows(np.arange(p.shape[0] + nchief))
    s.close()
    D = np.linalg.norm(p.max(0) - p.min(0))
    assert np.linalg.norm(A - A0) <= (1e-14 + 1e-15 * k * D) * np.linalg.norm(A0)


@pytest.mark.parametrize("nchief", [0, 5])
@pytest.mark.parametrize("method", ["gmres", "cgls", "block"])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 8, 9, 17])
def test_fp64_right_hand_sides(R, method, nchief):
    m = bem.Mesh().icosphere(2, 0.1)
    m.set_bc(0, 1, 0)
    if nchief:
        m.set_chief(C.ball_points(4, nchief, 0.04))
    k = 9.0
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP64)
    dirs = C.sphere_points(5 + R, R, 1.0)
    s.set_rhs(bem.RHS_PLANE, dirs, 1.0)
    s.solve({"gmres": bem.SOLVE_GMRES, "cgls": bem.SOLVE_CGLS, "block": bem.SOLVE_BLOCK_CG}[method], restart=60,
            tol=1e-8, maxit=4000, refine_tol=1e-12, max_refine=50)
    X = s.solution()
    A = s.rows(np.arange(m.num_pnts + nchief))
    s.close()
    x = np.vstack([m.pnts(), m.chief()]).astype(np.float64)
    B = np.exp(-1j * k * x @ dirs.astype(np.float64).T)
    X0 = np.linalg.lstsq(A, B, rcond=None)[0]
    assert np.linalg.norm(X - X0) <= (1e-8 if nchief else 1e-10) * np.linalg.norm(X0)
