"""bem_request_footprint against what a request allocates: an upper bound, and not
one that counts arrays of the other precision."""
import ctypes

import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem
import bemcases as C

METHODS = {"gmres": bem.SOLVE_GMRES, "cgls": bem.SOLVE_CGLS, "block": bem.SOLVE_BLOCK_CG, "qr": bem.SOLVE_QR}


# at 2562 nodes the assembly keeps more than N side columns of M entries
def test_footprint_counts_one_precision():
    N, E = 2562, 5120
    M = N + 16
    ld = (M + 63) // 64 * 64
    f = [bem.request_footprint(M, N, E, 1, precision=p, method=bem.SOLVE_CGLS) for p in (bem.PREC_FP32, bem.PREC_FP64)]
    assert f[1] - f[0] >= 8.0 * ld * N + 8.0 * ld * N


# the FP64 QR solves its right-hand sides together, with 2 x 256 doubles for each
# of the 41 workgroups
def test_footprint_of_fp64_qr_solves():
    f = [bem.request_footprint(2578, 2562, 5120, R, precision=bem.PREC_FP64, method=bem.SOLVE_QR) for R in (1, 64)]
    ld = 2624
    assert f[1] - f[0] >= 63 * (40 * ld + 8 * 2 * 256 * 41 + 16 * 2562)


class Pool:
    """Peak use of the device's memory pool."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.pool = ctypes.c_void_p()
        assert self.hip.hipDeviceGetDefaultMemPool(ctypes.byref(self.pool), 0) == 0

    def _attr(self, what):
        v = ctypes.c_uint64()
        assert self.hip.hipMemPoolGetAttribute(self.pool, what, ctypes.byref(v)) == 0
        return v.value

    def start(self):
        zero = ctypes.c_uint64(0)
        assert self.hip.hipMemPoolSetAttribute(self.pool, 8, ctypes.byref(zero)) == 0  # hipMemPoolAttrUsedMemHigh
        self.base = self._attr(7)  # hipMemPoolAttrUsedMemCurrent

    def peak(self):
        return self._attr(8) - self.base


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("subdiv,nchief,R,method", [
    (s, c, R, method) for s, c, R in ((3, 8, 1), (3, 8, 64), (4, 0, 3), (4, 16, 17), (5, 16, 4)) for method in METHODS
    if s < 5 or method != "qr"])
def test_footprint_bounds_the_pool(subdiv, nchief, R, method, precision):
    prec = bem.PREC_FP64 if precision == 64 else bem.PREC_FP32
    m = bem.Mesh().ellipsoid(subdiv, (0.075, 0.09, 0.11), nbumps=4, lmax=4, amp=0.03, seed=7)
    m.set_bc(0, 1, 0)
    if nchief:
        m.set_chief(C.ball_points(3, nchief, 0.03))
    bound = bem.request_footprint(m.num_pnts + nchief, m.num_pnts, m.num_elems, R, precision=prec,
                                  method=METHODS[method], restart=30)
    pool = Pool()
    pool.start()
    s = bem.Solver(m)
    s.assemble(9.0, prec)
    s.set_rhs(bem.RHS_PLANE, C.sphere_points(5 + R, R, 1.0), 1.0)
    s.solve(METHODS[method], restart=30, tol=1e-6, maxit=60, refine_tol=1e-8, max_refine=4)
    X = s.solution()
    peak = pool.peak()
    s.close()
    print("case: %d nodes, %d, %s, FP%d: peak %.1f MB, footprint %.1f MB" %
          (m.num_pnts, R, method, precision, peak / 1e6, bound / 1e6), flush=True)
    assert np.isfinite(X).all()
    assert 0 < peak <= bound
