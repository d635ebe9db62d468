"""Phases of far entries of the FP32 matrix where the body spans many radians: no
error common to them, which a solution would not average out.

Tolerances: an entry is a sum of a few elements' terms, each a product of a
handful of FP32 factors: four roundings (2.4e-7) in the root mean square, and the
mean of the errors' phases within one (6e-8).
"""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem

pytestmark = pytest.mark.gpu


# 44 and 20 radians across the body, elements of up to 0.5 and 0.2 radians (the
# rules of 12 and 16, and of 7 points)
@pytest.mark.parametrize("k", [220.0, 100.0])
@pytest.mark.parametrize("bc", [(0, 1, 0), (0.5 + 0.25j, 1.0 - 0.5j, 0.0)], ids=["rigid", "impedance"])
def test_far_entries_have_no_common_phase_error(k, bc):
    m = bem.Mesh().icosphere(5, 0.1)
    m.set_bc(*bc)
    rows = np.arange(7, m.num_pnts, 97)
    A = []
    for prec in (bem.PREC_FP32, bem.PREC_FP64):
        s = bem.Solver(m)
        s.assemble(k, prec)
        A.append(s.rows(rows))
        s.close()
    p = m.pnts().astype(np.float64)
    far = np.linalg.norm(p[rows][:, None] - p[None], axis=2) > 0.07  # 20 node spacings
    D, B = (A[0] - A[1])[far], A[1][far]
    rel = (D * B.conj()).sum() / (np.abs(B) ** 2).sum()
    rms = np.linalg.norm(D) / np.linalg.norm(B)
    print("case: k %g: mean %.2g%+.2gi, rms %.2g" % (k, rel.real, rel.imag, rms), flush=True)
    assert rms <= 2.4e-7
    assert abs(rel.imag) <= 6e-8
