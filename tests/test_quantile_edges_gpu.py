"""Quantile thresholds (device order statistics) against the oracle's definition at the edges of their kernels:
rows shorter than a thread's bins, partial groups, one and several block columns, counts from 1 to all but one
value, planes whose values share their leading bits or are zero, and spill lists that the first bound overflows
(the host then bisects).  Exact: the order statistics are FP32 values and the interpolation is FP64.
"""

import numpy as np
import pytest

from fdas_amd.host import FDAS
from oracle import fdas_oracle as O

from test_gpu_parity import PARTS, make

pytestmark = pytest.mark.gpu


def check(fop, n_harmonics, n_cands, part=FDAS.AllAccelerations, **kw):
    T, n = fop.shape
    f = make(n, n_templates=T, n_harmonics=n_harmonics, cands_per_harmonic=64, **kw)
    assert f.inject_FOP(fop.reshape(-1), FDAS.A), f.last_error
    rows = O.part_rows(T, PARTS[part])
    ref = O.quantile_thresholds(O.harmonic_planes(fop, n_harmonics, rows, dtype=np.float32), n_cands, rows)
    for _ in range(2):  # the workspace is kept between calls
        thr = f.quantile_thresholds(n_cands, part, FDAS.A)
        assert thr is not None, f.last_error
        assert np.array_equal(thr, ref)
    f.close()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 255, 513, 2049, 4099])
@pytest.mark.parametrize("n_harmonics,part", [(1, FDAS.AllAccelerations), (5, FDAS.NegativeAccelerations),
                                              (16, FDAS.PositiveAccelerations)])
def test_quantile_row_lengths(n, n_harmonics, part):
    fop = np.random.default_rng(n).exponential(size=(33, n)).astype(np.float32)
    M = len(O.part_rows(33, PARTS[part])) * n
    for n_cands in {1, min(20, M - 1), M // 2, M - 1} - {0}:
        check(fop, n_harmonics, n_cands, part)


@pytest.mark.parametrize("kind", ["narrow", "integers", "zeros"])
def test_quantile_value_distributions(kind):
    rng = np.random.default_rng(5)
    fop = {"narrow": 1.0 + 1e-6 * rng.random((9, 3000)), "integers": rng.integers(0, 4, (9, 3000)),
           "zeros": np.where(rng.random((9, 3000)) < 0.001, 3.0, 0.0)}[kind].astype(np.float32)
    for n_cands in (3, 100, 5000):
        check(fop, 4, n_cands)


@pytest.mark.parametrize("spill", [400, 3000])
def test_quantile_bisects_when_the_bound_overflows(spill):
    """Few blocks (no bound) or a block full of strong values: the first pass spills more than the lists hold."""
    rng = np.random.default_rng(spill)
    fop = rng.exponential(size=(9, 5000)).astype(np.float32)
    fop[4, 512:768] += 50.0
    for n_cands in (5, 200):
        check(fop, 8, n_cands, spill_per_harmonic=spill)


def test_quantile_ties_beyond_the_spill():
    f = make(4000, n_templates=9, n_harmonics=2, cands_per_harmonic=64, spill_per_harmonic=500)
    assert f.inject_FOP(np.ones(9 * 4000, np.float32), FDAS.A)
    assert f.quantile_thresholds(10, FDAS.AllAccelerations, FDAS.A) is None
    assert f.last_status == 7  # FDAS_EOVERFLOW
    f.close()
