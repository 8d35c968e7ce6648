"""The end of a summing workgroup, where it writes its staged hits: 1 to 16 planes (one to four planes per wave),
hits in one wave or in all, and 1, 8, 9 and many staged groups per plane.  Lists are exact against the oracle.
"""

import numpy as np
import pytest

from test_select_edges_gpu import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1, 2, 3, 4, 5, 8, 13, 16])
@pytest.mark.parametrize("groups", [1, 8, 9, 23, 24, 200])
def test_staged_groups(H, groups):
    """`groups` groups of 8 bins hold hits, in the first wave's 512 bins as long as they fit there, in every plane."""
    T, n = 3, 2500
    rng = np.random.default_rng(100 * H + groups)
    fop = (0.01 * rng.random((T, n))).astype(np.float32)
    at = 8 * rng.permutation(64 if groups <= 64 else n // 8)[:groups] + rng.integers(0, 8, min(groups, n // 8))
    fop[1, at] = 4.0 + rng.random(at.size).astype(np.float32)
    thr = np.full(H, 3.5, np.float32)
    det = run(fop, thr, 512)
    assert int(det[0]) == groups


@pytest.mark.parametrize("n", [7, 8, 511, 512, 513, 2047, 2048, 2049])
def test_hits_in_every_wave(n):
    rng = np.random.default_rng(n)
    fop = rng.exponential(size=(5, n)).astype(np.float32)
    run(fop, np.array([2.0, 4.0, 5.0, 6.0, 7.0], np.float32), 256)
