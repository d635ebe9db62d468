"""Rows of the matrix for collocation points on and next to the surface, entry by
entry, against the 36-point rule in extended precision.

Tolerance: u is the unit roundoff (6e-8, 1.1e-16), A the size |p_3 - x| + |e_1| +
|e_2| that the coordinates of a quadrature point's distance are formed from, r
its length.  Differences of coordinates are off by at most 4 u A, so 1 / r^3 by
12 u A / r; another 16 u cover the roundings of a term and its sums, 2 u k r its
phase; and the normal distance is off by 2 u A.  An entry may be off by the sum
of this over its points.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C
import oracle_py as orc

AIR = dict(dens=float(np.float32(1.2041)), speed=float(np.float32(343.21)))
L = np.longdouble


def _rows(p, elems, bc, k, xs, u):
    """(entries, tolerances) of the rows xs (no nodes), C x N."""
    gp, gw = (v.astype(L) for v in np.polynomial.legendre.leggauss(6))
    for _ in range(2):  # to extended precision: Newton on P_6
        P6, P5 = (np.polynomial.legendre.legval(gp, [0] * d + [1]) for d in (6, 5))
        d6 = 6 * (gp * P6 - P5) / (gp * gp - 1)
        gp = gp - P6 / d6
    P6, P5 = (np.polynomial.legendre.legval(gp, [0] * d + [1]) for d in (6, 5))
    d6 = 6 * (gp * P6 - P5) / (gp * gp - 1)
    gw = 2 / ((1 - gp * gp) * d6 * d6)
    th, rho = (v.ravel() for v in np.meshgrid((1 + gp) / 2, (1 + gp) / 2, indexing="ij"))
    W = (np.outer(gw, gw).ravel() / 4) * rho
    Nq = np.stack([rho * (1 - th), rho * th, 1 - rho])  # 3 x 36
    t = p[elems].astype(L)
    e1, e2 = t[:, 0] - t[:, 2], t[:, 1] - t[:, 2]
    cr = np.cross(e1, e2)
    J = np.sqrt((cr * cr).sum(1))
    n = cr / J[:, None]
    y = np.einsum("jq,ejd->eqd", Nq, t)
    beta = L(1) * complex(bc[0]) / complex(bc[1])
    rw = L(AIR["dens"]) * L(k) * L(AIR["speed"])
    out = np.zeros((len(xs), len(p)), np.clongdouble)
    tol = np.zeros((len(xs), len(p)), L)
    k = L(k)
    for i, x in enumerate(xs.astype(L)):
        a = t[:, 2] - x
        dn = (n * a).sum(1)[:, None]
        A = (np.sqrt((a * a).sum(1)) + np.sqrt((e1 * e1).sum(1)) + np.sqrt((e2 * e2).sum(1)))[:, None]
        r = np.sqrt(((y - x) ** 2).sum(2))
        ex = (np.cos(k * r) - 1j * np.sin(k * r)) * W * (J / (4 * L(np.pi)))[:, None]
        h = -dn * ex * (1 / r ** 3 + 1j * k / r ** 2)
        g = 1j * rw * ex / r
        loose = u * (16 + 12 * A / r + 2 * k * r)
        th_ = np.abs(h) * loose + 2 * u * A * np.abs(ex) * (1 / r ** 3 + k / r ** 2) + np.abs(beta * g) * loose
        for j in range(3):
            np.add.at(out[i], elems[:, j], ((h - beta * g) * Nq[j]).sum(1))
            np.add.at(tol[i], elems[:, j], (th_ * Nq[j]).sum(1))
    return out, tol


def test_reference_matches_oracle():
    orc.quad_init(6)
    m = bem.Mesh().icosphere(1, 0.1)
    m.set_bc(0.5 + 0.25j, 1.0 - 0.5j, 0.0)
    p, e, bcs = C.mesh_arrays(m)
    xs = C.ball_points(5, 4, 0.06)
    A0, _ = orc.assemble(20.0, np.vstack([p, xs]).astype(np.float64), len(p), e, bcs, dtype=np.float64, **AIR)
    A, tol = _rows(p, e, (0.5 + 0.25j, 1.0 - 0.5j), 20.0, xs, 1.1e-16)
    assert np.all(np.abs(A0[len(p):] - A) <= 2 * tol)


def _matrix_rows(m, xs, k, prec):
    """The rows xs as CHIEF rows of the assembled system."""
    m.set_chief(xs)
    s = bem.Solver(m)
    s.assemble(k, prec)
    A = s.rows(np.arange(m.num_pnts, m.num_pnts + len(xs)))
    s.close()
    return A


def _octahedron(n):
    """Nodes and triangles of an octahedron, every face cut into n^2 triangles,
    whose centroids are whole numbers (coordinates are multiples of 3)."""
    at, e = {}, []
    for sx in (1, -1):
        for sy in (1, -1):
            for sz in (1, -1):
                v = lambda i, j: at.setdefault((3 * sx * i, 3 * sy * j, 3 * sz * (n - i - j)), len(at))
                for i in range(n):
                    for j in range(n - i):
                        t = [(v(i, j), v(i + 1, j), v(i, j + 1))]
                        if i + j < n - 1:
                            t.append((v(i + 1, j), v(i + 1, j + 1), v(i, j + 1)))
                        e += [q if sx * sy * sz < 0 else q[::-1] for q in t]
    return np.array(list(at), np.float32), np.array(e, np.int32)


# rows at zero distance from the centroids of elements (6 nodes take the halo plan
# and its kernels, 66 and 258 the element-once plan)
@pytest.mark.gpu
@pytest.mark.parametrize("prec,u", [(bem.PREC_FP32, 6e-8), (bem.PREC_FP64, 1.1e-16)], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n,k", [(1, 0.1), (4, 0.0), (4, 0.1), (8, 1.0)])
def test_row_at_a_centroid(prec, u, n, k):
    p, e = _octahedron(n)
    m = bem.Mesh().set(p, e, (0.5 + 0.25j, 1.0 - 0.5j, 0.0))
    xs = np.concatenate([p[e[::5]].mean(1), [(0.5, 0.25, 0)]]).astype(np.float32)
    assert np.array_equal(xs[:-1], np.rint(xs[:-1]))
    A = _matrix_rows(m, xs, k, prec)
    A0, tol = _rows(p, e, (0.5 + 0.25j, 1.0 - 0.5j), float(np.float32(k)), xs, u)
    assert np.all(np.abs(A - A0) <= tol)


def _body(subdiv, bc):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=8, lmax=6, amp=0.05, seed=70 + subdiv)
    m.set_bc(*bc, 0.0)
    return m


def _above(p, elems, height, count):
    """Points over quadrature points of some elements, `height` edges off, on
    either side in turn."""
    gp = np.polynomial.legendre.leggauss(6)[0]
    sel = np.linspace(0, len(elems) - 1, count).astype(int)
    t = p[elems[sel]].astype(np.float64)
    th, rho = (1 + gp[np.arange(count) % 6]) / 2, (1 + gp[np.arange(count) // 2 % 6]) / 2
    y = t[:, 0] * (rho * (1 - th))[:, None] + t[:, 1] * (rho * th)[:, None] + t[:, 2] * (1 - rho)[:, None]
    n = np.cross(t[:, 0] - t[:, 2], t[:, 1] - t[:, 2])
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    edge = np.linalg.norm(t[:, 0] - t[:, 1], axis=1)[:, None]
    side = np.where(np.arange(count) % 2, -1.0, 1.0)[:, None]
    return (y + side * height * edge * n).astype(np.float32)


# a mesh on the element-once plan of few rows, and one past 4e6 pairs; elements
# within and past the phase limit of the FP64 kernel (k rho 0.79)
@pytest.mark.gpu
@pytest.mark.parametrize("prec,u", [(bem.PREC_FP32, 6e-8), (bem.PREC_FP64, 1.1e-16)], ids=["fp32", "fp64"])
@pytest.mark.parametrize("bc", [(0, 1), (0.5 + 0.25j, 1.0 - 0.5j)], ids=["rigid", "impedance"])
@pytest.mark.parametrize("subdiv,k", [(2, 9.0), (2, 90.0), (4, 30.0)])
@pytest.mark.parametrize("height", [0.3, 0.1, 0.03, 0.01])
def test_rows_next_to_the_surface(height, subdiv, k, bc, prec, u):
    m = _body(subdiv, bc)
    p, e, _ = C.mesh_arrays(m)
    xs = _above(p, e, height, 12)
    A = _matrix_rows(m, xs, k, prec)
    A0, tol = _rows(p, e, bc, float(np.float32(k)), xs, u)
    ratio = np.abs(A - A0) / tol
    print("case: height %g: worst %.2g of the tolerance, median %.2g" % (height, ratio.max(), np.median(ratio)), flush=True)
    assert ratio.max() <= 1


# the rows of a radiation operator, on the small mesh's tiles
@pytest.mark.gpu
@pytest.mark.parametrize("height", [0.3, 0.1, 0.03, 0.01])
def test_operator_rows_next_to_the_surface(height):
    m = _body(2, (0, 1))
    p, e, _ = C.mesh_arrays(m)
    xs = _above(p, e, height, 70)
    s = bem.Solver(m)
    s.assemble(9.0, bem.PREC_FP32)
    F = s.field_matrix(xs).get_field_matrix()
    s.close()
    F0, tol = _rows(p, e, (0, 1), 9.0, xs, 6e-8)
    assert np.all(np.abs(F - F0) <= tol)
