"""Candidate selection at the sizes where its workgroups change: caps around 1024 and 4096 (workgroup forms),
list lengths around 64-entry runs, detections just above the cap, pools of tied powers below and above the
counted size, and dense planes that overflow the compact list.  Lists are exact against the oracle.
"""

import numpy as np
import pytest

from fdas_amd.host import FDAS
from oracle import fdas_oracle as O

from test_gpu_parity import assert_lists_match, make, wide_by_plane

pytestmark = pytest.mark.gpu


def run(fop, thr, cap):
    T, n = fop.shape
    H = len(thr)
    f = make(n, n_templates=T, n_harmonics=H, cands_per_harmonic=cap)
    assert f.inject_FOP(fop.reshape(-1), FDAS.A), f.last_error
    assert f.perform_harmonic_summing(thr, FDAS.AllAccelerations, FDAS.A), f.last_error
    rows = O.part_rows(T, "all")
    sel = O.select(O.detect(O.harmonic_planes(fop, H, rows, dtype=np.float32), thr, rows), cap)
    planes, det = wide_by_plane(f, FDAS.A, H)
    assert_lists_match(planes, det, sel, thr, cap, T // 2, exact=True)
    f.close()
    return det


@pytest.mark.parametrize("cap", [1, 63, 65, 1024, 1025, 4096, 4097, 8192])
@pytest.mark.parametrize("share", [0.02, 0.5])  # of the bins above the threshold: few (no cut) / many
def test_select_caps(cap, share):
    rng = np.random.default_rng(cap)
    fop = rng.exponential(size=(33, 4999)).astype(np.float32)
    det = run(fop, np.array([-np.log(share), 2.0 - np.log(share)], np.float32), cap)
    assert det[0] > 0


@pytest.mark.parametrize("n_tied", [1, 500, 1024, 1025, 4096, 4097])
def test_select_tied_pool(n_tied):
    """n_tied bins share one power at the cut: the smallest keys among them are kept."""
    cap, T, n = 300, 9, 2048
    rng = np.random.default_rng(n_tied)
    fop = np.zeros(T * n, np.float32)
    at = rng.permutation(T * n)
    fop[at[:n_tied]] = 5.0
    fop[at[n_tied:n_tied + 200]] = 50.0 + np.arange(200, dtype=np.float32)
    fop[at[n_tied + 200:n_tied + 400]] = 2.0
    run(fop.reshape(T, n), np.array([1.0], np.float32), cap)


@pytest.mark.parametrize("extra", [0, 1, 63])
def test_select_just_above_cap(extra):
    cap, T, n = 1024, 9, 3001
    rng = np.random.default_rng(extra)
    fop = np.zeros(T * n, np.float32)
    fop[rng.permutation(T * n)[:cap + extra]] = (1.5 + rng.random(cap + extra)).astype(np.float32)
    det = run(fop.reshape(T, n), np.array([1.0], np.float32), cap)
    assert int(det[0]) == cap + extra
