"""Fields of many points, which the kernels may take in another order: every point's
value is the one it has in a call of its own, bit for bit, also where points are
far away, equal, infinite or not a number."""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu


# sorted from 4e6 pairs on: 320, 1280 and 5120 elements; below that, and with no point
# near the body
@pytest.mark.parametrize("subdiv,P,R,dist", [(2, 12499, 1, 1.1), (2, 12500, 2, 1.1), (3, 3125, 1, 1.02), (3, 9001, 17, 1.3),
                                             (4, 1000, 1, 1.05), (4, 2000, 3, 1.05), (4, 2000, 1, 30.0)])
def test_value_does_not_depend_on_the_order(subdiv, P, R, dist):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=4, lmax=4, amp=0.03, seed=3)
    m.set_bc(0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j).set_chief(C.ball_points(3, 5, 0.03))
    s = bem.Solver(m)
    s.assemble(9.0, bem.PREC_FP32)
    s.set_rhs(bem.RHS_PLANE, C.sphere_points(4 + R, R, 1.0), 1.0)
    s.solve(bem.SOLVE_CGLS, tol=1e-6, maxit=60, refine_tol=1e-6, max_refine=2)
    xs = C.sphere_points(6, P, 0.11 * dist)
    xs[::7] *= 5.0
    xs[10], xs[11] = xs[12], xs[12]
    if dist < 10:
        xs[100] = (np.inf, 0, 0)
        xs[200, 1] = np.nan
        xs[300] = 1e30
    f = s.field(xs)
    part = np.concatenate([s.field(xs[a:a + 700]) for a in range(0, P, 700)])
    s.close()
    assert np.array_equal(f.view(np.uint32), part.view(np.uint32))
    assert np.isfinite(f).all(axis=1).sum() >= P - 3
