"""Harmonic summing at the edges of its loads: row lengths around one thread's 8 bins, one wave's 512 and one
workgroup's 2048, so that the last group of a row is whole, partial or the whole row, in the plane's last row
and in rows before it.  Low thresholds let about a third of all bins through, the last ones among them; sums
are bit-exact against the FP32 oracle.
"""

import numpy as np
import pytest

from fdas_amd.host import FDAS
from oracle import fdas_oracle as O

from test_gpu_parity import PARTS, assert_lists_match, make, wide_by_plane

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 15, 16, 511, 513, 2047, 2049, 2063, 4097])
@pytest.mark.parametrize("n_templates,n_harmonics,part", [(1, 1, FDAS.AllAccelerations), (9, 8, FDAS.AllAccelerations),
                                                          (33, 4, FDAS.NegativeAccelerations),
                                                          (33, 16, FDAS.PositiveAccelerations)])
def test_hsum_row_length_edges(n, n_templates, n_harmonics, part):
    rng = np.random.default_rng(n * 31 + n_templates)
    fop = rng.exponential(1.0, size=(n_templates, n)).astype(np.float32)
    fop[:, -1] += 20.0  # the last bin of every row passes its threshold on every plane
    thr = np.array([k + 0.3 * np.sqrt(k) for k in range(1, n_harmonics + 1)], np.float32)
    f = make(n, n_templates=n_templates, n_harmonics=n_harmonics, cands_per_harmonic=4096)
    assert f.inject_FOP(fop.reshape(-1), FDAS.A), f.last_error
    assert f.perform_harmonic_summing(thr, part, FDAS.A), f.last_error
    rows = O.part_rows(n_templates, PARTS[part])
    sel = O.select(O.detect(O.harmonic_planes(fop, n_harmonics, rows, dtype=np.float32), thr, rows), 4096)
    planes, det = wide_by_plane(f, FDAS.A, n_harmonics)
    assert_lists_match(planes, det, sel, thr, 4096, n_templates // 2, exact=True)
    assert int(det[0]) >= len(rows)
    f.close()
