"""GPU test of single trials whose bank falls into many row groups of the FT convolution.  Up to 16 groups' job
descriptors travel as a kernel argument, more through a pinned array that an earlier launch's copy may still be reading.
Templates of 20 and of 600 taps alternate in blocks, so that each block is a group of its own: 16 of them (the most
that the argument holds), 22 and 43; and the longest drift bank, in 19 and 16."""

import numpy as np
import pytest

from fdas_amd import synth
from fdas_amd.host import FDAS
from oracle import fdas_oracle as O

from test_gpu_parity import FOP_TOL, bank_for, make, rel_err, spectrum

pytestmark = pytest.mark.gpu

N = 4999


def alternating_bank(block, n_templates=127, taps=(20, 600)):
    rng = np.random.default_rng(block)
    bank = np.zeros((n_templates, max(taps)), np.complex64)
    for t in range(n_templates):
        m = taps[t // block % 2]
        row = rng.standard_normal(m) + 1j * rng.standard_normal(m)
        bank[t, :m] = row / np.linalg.norm(row)
    return bank


@pytest.mark.parametrize("tile,block", [(1024, 2), (1024, 3), (2048, 6)])
def test_alternating_taps(tile, block):
    H, bank = 4, alternating_bank(block)
    f = make(N, n_templates=127, max_taps=600, tile=tile, n_harmonics=H, cands_per_harmonic=64)
    x, y = spectrum(N, 1), spectrum(N, 2)
    thr = synth.noise_thresholds(x, H)

    def state(ab):
        fop = np.zeros(f.get_fop_sz(), np.float32)
        lists = [np.zeros(f.get_candidate_list_sz(), t) for t in (np.uint32, np.float32)]
        assert f.retrieve_FOP(fop, ab) and f.retrieve_candidates(*lists, ab), f.last_error
        return [fop, *lists]

    # the blocking calls, whole bank and then the non-negative half again, against the oracle
    assert f.upload_template_taps(bank, FDAS.A) and f.upload_template_taps(bank, FDAS.B), f.last_error
    want = {}
    for which, s in (("x", x), ("y", y)):
        assert f.perform_input_tiling(s, FDAS.A) and f.perform_ft_convolution(2, FDAS.A), f.last_error
        assert f.perform_harmonic_summing(thr, 2, FDAS.A), f.last_error
        want[which] = state(FDAS.A)
        ref = O.fop_fft(s, bank)
        assert rel_err(want[which][0].reshape(127, N), ref) <= FOP_TOL
        # (the half's groups have overlaps of their own, so its FOP is rounded differently)
        assert f.perform_ft_convolution(1, FDAS.A), f.last_error
        assert rel_err(state(FDAS.A)[0].reshape(127, N), ref) <= FOP_TOL
    # launches enqueued over one another: the job array is rewritten while earlier launches are in flight
    out = [np.zeros(f.get_candidate_list_sz(), t) for t in (np.uint32, np.float32)]
    for order in ("xy", "yx", "xyyx", "yxxxy"):
        for i, s in enumerate(order):
            assert f.launch({"x": x, "y": y}[s], thr, *out, 1 if i == 0 else 2, FDAS.B), f.last_error
        assert f.wait(FDAS.B), f.last_error
        got = state(FDAS.B)
        assert all(np.array_equal(a, b) for a, b in zip(got, want[order[-1]]))
        assert np.array_equal(out[0], got[1]) and np.array_equal(out[1], got[2])
    f.close()


@pytest.mark.parametrize("tile", [1024, 2048])
def test_longest_drift_bank(tile):
    bank = bank_for(255, 600)
    f = make(N, n_templates=255, max_taps=600, tile=tile, n_harmonics=1, cands_per_harmonic=16)
    assert f.upload_template_taps(bank, FDAS.A), f.last_error
    x = spectrum(N, 3)
    assert f.perform_input_tiling(x, FDAS.A), f.last_error
    fop = np.zeros(f.get_fop_sz(), np.float32)
    for part in (0, 1, 2):
        assert f.perform_ft_convolution(part, FDAS.A), f.last_error
    assert f.retrieve_FOP(fop, FDAS.A), f.last_error
    assert rel_err(fop.reshape(255, N), O.fop_fft(x, bank)) <= FOP_TOL
    f.close()
