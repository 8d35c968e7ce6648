"""Candidate selection where planes move between the direct path (the last kernel reads the spill list itself: at most
cap + 4096 detections) and the histogram and compaction kernels, and at the run lengths of the sort of short lists.
Lists are exact against the oracle.
"""

import numpy as np
import pytest

from test_select_edges_gpu import run

pytestmark = pytest.mark.gpu


def plane(n_above, seed, T=33, n=4999):
    """T x n powers, n_above of them above 1, each another value."""
    rng = np.random.default_rng(seed)
    fop = np.zeros(T * n, np.float32)
    fop[rng.permutation(T * n)[:n_above]] = 1.001 + rng.permutation(n_above).astype(np.float32) * np.float32(1e-3)
    return fop.reshape(T, n)


@pytest.mark.parametrize("cap", [512, 1024, 2048])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_direct_limit(cap, extra):
    det = run(plane(cap + 4096 + extra, cap + extra), np.array([1.0], np.float32), cap)
    assert int(det[0]) == cap + 4096 + extra


@pytest.mark.parametrize("kept", [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 767, 1023, 1024])
def test_run_lengths(kept):
    thr = np.array([1.0], np.float32)
    assert int(run(plane(kept, kept), thr, 1024)[0]) == kept  # all detections kept
    assert int(run(plane(3000, kept), thr, kept)[0]) == 3000  # a cut at `kept`


def test_direct_with_equal_powers_beyond_the_pool():
    """Every detection has one power: the cut bin holds them all, more than the pool's 4096 at a cap of 600."""
    rng = np.random.default_rng(3)
    fop = np.zeros(33 * 4999, np.float32)
    fop[rng.permutation(fop.size)[:4650]] = 3.0
    run(fop.reshape(33, 4999), np.array([1.0], np.float32), 600)
