"""Which iteration and which products block CG takes by the size of the system:
the lockstep CG (its result bit for bit) where the block does not pay, the block
on FP32 products (the result with BEM_GEMM_NO_F16, bit for bit) for few right-hand
sides below 4e8 of M N nrhs, on FP16-split products from there on.
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

pytestmark = pytest.mark.gpu

KW = dict(tol=1e-6, maxit=6000, refine_tol=1e-10, max_refine=50)


def _sphere(rings, cols):
    """A sphere of rings x cols + 2 nodes on circles of latitude."""
    t = np.pi * np.arange(1, rings + 1) / (rings + 1)
    f = 2 * np.pi * np.arange(cols) / cols
    p = np.stack([np.outer(np.sin(t), np.cos(f)), np.outer(np.sin(t), np.sin(f)),
                  np.outer(np.cos(t), np.ones(cols))], axis=-1).reshape(-1, 3)
    p = np.concatenate([p, [(0, 0, 1), (0, 0, -1)]]) * 0.1
    a = np.arange(cols)
    b = (a + 1) % cols
    e = [np.stack([a * 0 + rings * cols, b, a], 1), np.stack([a * 0 + rings * cols + 1, a, b], 1) + [0, 1, 1] * np.array(
        (rings - 1) * cols)]
    for r in range(rings - 1):
        u, v = a + r * cols, b + r * cols
        e += [np.stack([u, v, v + cols], 1), np.stack([u, v + cols, u + cols], 1)]
    return p.astype(np.float32), np.concatenate(e).astype(np.int32)


def _solver(rings, cols, R):
    p, e = _sphere(rings, cols)
    m = bem.Mesh().set(p, e, (0, 1, 0)).set_chief(C.ball_points(11, 16, 0.05))
    s = bem.Solver(m)
    s.assemble(16.0, bem.PREC_FP32)
    s.set_rhs(bem.RHS_PLANE, C.sphere_points(50 + R, R, 1.0), 1.0)
    return s


def _solve(s, method):
    st = s.solve(method, **KW)
    assert st["converged"] == 1
    return s.solution(), st["iterations"]


# each rule's limit missed alone: M N nrhs 1.05e8; 1.69e8 with M N 1.06e7; 1.13e8
# with M N 1.6e7; more than 16 right-hand sides below 4e8
@pytest.mark.parametrize("rings,cols,R", [(40, 64, 16), (45, 72, 16), (50, 80, 7), (50, 80, 17)])
def test_small_systems_take_the_lockstep_iteration(rings, cols, R):
    s = _solver(rings, cols, R)
    X, it = _solve(s, bem.SOLVE_BLOCK_CG)
    Xl, itl = _solve(s, bem.SOLVE_CGLS)
    s.close()
    assert it == itl and np.array_equal(X, Xl)


# M N nrhs 1.29e8, 2.57e8, 3.97e8 and 4.08e8
@pytest.mark.parametrize("rings,cols,R,split", [(50, 80, 8, False), (50, 80, 16, False), (70, 90, 10, False),
                                                (71, 90, 10, True)])
def test_products_of_the_block(monkeypatch, rings, cols, R, split):
    s = _solver(rings, cols, R)
    X, it = _solve(s, bem.SOLVE_BLOCK_CG)
    Xl, itl = _solve(s, bem.SOLVE_CGLS)
    monkeypatch.setenv("BEM_GEMM_NO_F16", "1")
    X32, _ = _solve(s, bem.SOLVE_BLOCK_CG)
    s.close()
    assert it < itl
    assert np.array_equal(X, X32) != split
    # both to 1e-10 on the normal equations of a matrix with a condition number of
    # a few hundred
    assert np.linalg.norm(X - Xl) <= 1e-5 * np.linalg.norm(Xl)
