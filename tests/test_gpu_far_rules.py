"""The far rules of the FP32 assembly (far_rules.hpp): fewer quadrature points for
the elements that every row of a wave is far from, against the FP64 oracle's
36-point rule, across the rules' limits in distance and in elements per
wavelength, and the same for the field operator's rows.

Tolerance (Frobenius, relative): the rules differ from the 36 points by at most
3.3e-8; an entry is a sum over about 6 elements of FP32 terms, each a product of
a few roundings of 6e-8, so 3e-7; and the phase k r is rounded to 6e-8 k r on the
36-point path, with r at most the diameter D: 3e-7 + 6e-8 k D.
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


def oracle(mesh, k, chief):
    p, e, bc = C.mesh_arrays(mesh)
    M = p.shape[0] + chief.shape[0]
    A, B = orc.assemble(float(np.float32(k)), np.vstack([p, chief]).astype(np.float64), p.shape[0], e, bc,
                        np.zeros((M, 1), complex), dtype=np.float64, **AIR)
    return A, np.asarray(B).reshape(M, -1)


def diameter(p):
    return float(np.linalg.norm(p.max(0) - p.min(0)))


# elements seen at most 5, 20, 40 and 80 rho away; kappa = k rho about 0, 0.2
# (7-point limit), 0.55 (12- and 16-point limit) and 0.9 (36 points everywhere);
# CHIEF counts that leave full, partial and empty waves
@pytest.mark.parametrize("bc", [(0, 1, 0), (0, 1, -1), (0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j)],
                         ids=["rigid", "source", "impedance"])
@pytest.mark.parametrize("subdiv,kappa,nchief", [(1, 0.1, 0), (2, 0.2, 1), (3, 0.01, 62), (3, 0.23, 63), (3, 0.55, 7),
                                                 (3, 0.9, 8), (4, 0.05, 16), (4, 0.21, 62), (4, 0.58, 254)])
def test_far_rules_match_oracle(subdiv, kappa, nchief, bc):
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=8, lmax=6, amp=0.05, seed=40 + subdiv)
    m.set_bc(*bc)
    chief = C.ball_points(77, nchief, 0.03) if nchief else np.zeros((0, 3), np.float32)
    if nchief:
        m.set_chief(chief)
    p, e, _ = C.mesh_arrays(m)
    cen = p[e].mean(1)
    rho = np.median(np.linalg.norm(p[e] - cen[:, None], axis=2).max(1))
    k = kappa / rho
    A0, B0 = oracle(m, k, chief)
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP32)
    s.set_rhs(bem.RHS_PLANE, [[0, 0, 1]], 0.0)
    A, B = s.system()
    s.close()
    tol = 3e-7 + 6e-8 * k * diameter(p)
    assert np.linalg.norm(A - A0) <= tol * np.linalg.norm(A0)
    assert np.linalg.norm(B - B0) <= tol * np.linalg.norm(B0) if np.any(B0) else not np.any(B)


# rows at the rules' distances from every element (both sides of each limit),
# and far enough that k r passes 256 revolutions
@pytest.mark.parametrize("dist", [1.2, 2.0, 6.0, 900.0])
@pytest.mark.parametrize("P", [1, 63, 65, 300])
def test_far_rules_field_rows(dist, P):
    m = bem.Mesh().ellipsoid(3, (0.075, 0.09, 0.11), nbumps=8, lmax=6, amp=0.05, seed=9)
    m.set_bc(0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j)
    p, e, bc = C.mesh_arrays(m)
    k = 30.0
    xs = C.sphere_points(5, P, 0.115 * dist)
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP32)
    F = s.field_matrix(xs).get_field_matrix()
    s.close()
    F0 = orc.assemble_rows(k, np.vstack([p, xs]).astype(np.float64), p.shape[0], e, bc, p.shape[0], p.shape[0] + P,
                              dtype=np.float64, **AIR)
    tol = 3e-7 + 6e-8 * k * (0.115 * dist + 0.13)
    assert np.linalg.norm(F - F0) <= tol * np.linalg.norm(F0)


# an element-once plan of a handful of nodes per tile: some nodes' own tiles
# write nothing to their columns; the same matrix as in few tiles up to the
# order of the sums (6 terms of an entry, 6e-8 each)
@pytest.mark.parametrize("tiles", ["4", "40", "160", "300"])
def test_small_tiles_match_oracle(tiles, monkeypatch):
    monkeypatch.setenv("BEM_TILES", tiles)
    m = bem.Mesh().icosphere(3, 0.1)
    m.set_bc(0, 1, -1)
    k = 3.0
    A0, _ = oracle(m, k, np.zeros((0, 3), np.float32))
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP32)
    A, _ = s.system()
    s.close()
    assert np.linalg.norm(A - A0) <= (3e-7 + 6e-8 * k * 0.35) * np.linalg.norm(A0)


# the direct field kernel: P around a wave, R around its passes of 1, 4 and 16,
# points next to the surface (36 points) and far from it, against the oracle
# with the same solutions.  The terms an FP32 sum over the elements adds, and
# so its roundings, have the size int |dG/dn| |p| + rho omega int |G| (|beta| |p|
# + |gamma|): up to 2 max|p| of the first (twice the solid angle of a closed
# surface), the second from the elements' areas and distances.
@pytest.mark.parametrize("bc", [(0, 1, 0), (0.5 + 0.25j, 1.0 - 0.5j, 0.3 + 0.1j)], ids=["rigid", "impedance"])
@pytest.mark.parametrize("P,R", [(1, 1), (63, 2), (64, 4), (65, 5), (7, 16), (130, 17)])
@pytest.mark.parametrize("dist", [1.03, 1.5, 8.0])
def test_field_points_by_term_size(P, R, dist, bc):
    m = bem.Mesh().icosphere(2, 0.1)
    m.set_bc(*bc)
    p, e, bcs = C.mesh_arrays(m)
    k = 11.0
    dirs = C.sphere_points(31, R, 1.0)
    s = bem.Solver(m)
    s.assemble(k, bem.PREC_FP32)
    s.set_rhs(bem.RHS_PLANE, dirs, 1.0)
    s.solve(bem.SOLVE_QR)
    x = s.solution()
    xs = C.sphere_points(32, P, 0.1 * dist)
    out = s.field(xs)
    one = s.field(xs[:1])
    s.close()
    x64 = xs.astype(np.float64)
    inc = np.exp(-1j * k * x64 @ dirs.astype(np.float64).T)
    f0 = orc.field(k, p.astype(np.float64), p.shape[0], e, bcs, x64, x, inc=inc, dtype=np.float64, **AIR)
    f0 = np.asarray(f0).reshape(P, R)
    tri = p[e].astype(np.float64)
    area = np.linalg.norm(np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]), axis=1) / 2
    G = (area / (4 * np.pi * np.linalg.norm(x64[:, None] - tri.mean(1)[None], axis=2))).sum(1)[:, None]
    beta, gamma, rw = abs(bc[0] / bc[1]), abs(bc[2] / bc[1]), AIR["dens"] * k * AIR["speed"]
    size = (2 + rw * G * beta) * np.abs(x).max(0)[None] + rw * G * gamma + np.abs(inc)
    assert np.all(np.abs(out - f0) <= (3e-7 + 6e-8 * k * 0.1 * (dist + 1)) * size)
    assert np.array_equal(out[:1], one)  # a point's value does not depend on the others
