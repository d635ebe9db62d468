"""The assembly's launch shape is the one of the time a problem is built, also
where its tiles are made later, and the tuner's default is what a build without
a tuned shape runs."""
import numpy as np
import pytest

import bem_gpu_clean_cpp_amd as bem

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def clear():
    bem.tune_clear()
    yield
    bem.tune_clear()


def _buckets(m):
    return [int(np.rint(2 * np.log2(v))) for v in (m.num_pnts, m.num_elems)]


def _assembled(s):
    s.assemble(7.0, bem.PREC_FP32)
    return s.rows(np.arange(0, 642, 5))


# 512 waves: 13 tiles of 642 nodes; without a tuned shape 80.  The sums of a
# row's tiles are rounded in tile order, so the diagonal tells them apart.
def test_tiles_are_those_of_the_build(tmp_path):
    m = bem.Mesh().icosphere(3, 0.1)
    f = tmp_path / "tune"
    f.write_text("%d %d 4 512\n" % tuple(_buckets(m)))
    bem.tune_load(f)
    s = bem.Solver(m)
    A = _assembled(s)
    s.close()
    f.write_text("%d %d 4 32768\n" % tuple(_buckets(m)))
    bem.tune_load(f)
    s = bem.Solver(m)
    other = _assembled(s)
    s.close()
    assert not np.array_equal(A, other)
    f.write_text("%d %d 4 512\n" % tuple(_buckets(m)))
    bem.tune_load(f)
    s = bem.Solver(m)  # built with 512 waves, assembled after they are gone
    bem.tune_clear()
    B = _assembled(s)
    s.close()
    assert np.array_equal(A, B)


# all shapes with one lane a row have the same tiles at this size, so the
# default is about as fast as the best (the kernels of four lanes a row take
# several times as long in FP64)
@pytest.mark.parametrize("precision", [32, 64])
def test_default_is_the_untuned_build(precision):
    m = bem.Mesh().icosphere(3, 0.1)
    r = bem.autotune_assembly(m, 7.0, bem.PREC_FP64 if precision == 64 else bem.PREC_FP32)
    print("case:", r, flush=True)
    assert 0 < r["best_ms"] <= r["default_ms"] <= 2 * r["best_ms"]
