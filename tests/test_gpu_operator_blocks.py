"""A radiation operator of many points is assembled in blocks of rows: the same
rows bit for bit as in an operator of those points alone, and memory beside the
operator that does not grow with their number."""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C
from test_gpu_footprint import Pool

pytestmark = pytest.mark.gpu


def _body(subdiv):
    return bem.Mesh().icosphere(subdiv, 0.1).set_bc(0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j)


# 642 nodes: blocks of at most 13312 rows; 162 nodes: 52480.  One block less a row,
# a row more, several of them
@pytest.mark.parametrize("subdiv,P", [(3, 13311), (3, 13312), (3, 13313), (3, 40001), (2, 52481)])
def test_rows_of_the_blocks(subdiv, P):
    m = _body(subdiv)
    xs = C.sphere_points(5, P, 0.4)
    s = bem.Solver(m)
    s.assemble(9.0, bem.PREC_FP32)
    F = s.field_matrix(xs).get_field_matrix()
    s.set_rhs(bem.RHS_PLANE, [[0, 0, 1.0]], 1.0)
    s.solve(bem.SOLVE_QR)
    f = s.field_apply()
    first = [0, P - 200] + [b for b in range(6400, P - 1000, 6400)]
    for a in first:
        a = a // 64 * 64  # the rows of a wave take the same rule
        part = xs[a:a + 320]
        assert np.array_equal(s.field_matrix(part).get_field_matrix(), F[a:a + 320])
        # (the product over the operator sums in another order: 642 terms)
        d = s.field_apply() - f[a:a + 320]
        assert np.linalg.norm(d) <= 6e-8 * np.sqrt(642) * np.linalg.norm(f[a:a + 320])
    s.close()


@pytest.mark.parametrize("subdiv,P", [(3, 100000), (4, 60000)])
def test_memory_beside_the_operator(subdiv, P):
    m = _body(subdiv)
    s = bem.Solver(m)
    s.assemble(9.0, bem.PREC_FP32)
    bem.sync()
    pool = Pool()
    pool.start()
    s.field_matrix(C.sphere_points(6, P, 0.4))
    peak = pool.peak()
    s.close()
    rows = 8.0 * m.num_pnts * P
    print("case: operator %.0f MB, peak %.0f MB" % (rows / 1e6, peak / 1e6), flush=True)
    # 8192 workgroups of 256 rows over the tiles of at least 4 (642 nodes) or 8
    # nodes; 2 N side columns and the partials, 1.5 columns a tile; the points
    tiles = m.num_pnts // 4 if m.num_pnts < 1000 else m.num_pnts // 8
    assert peak <= rows + 8.0 * 256 * (8192 / tiles + 1) * (2 * m.num_pnts + 1.5 * tiles) + 100.0 * P + 1e7
