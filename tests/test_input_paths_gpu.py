"""GPU test of the ways a spectrum reaches the single-trial path, and of its device times.

Small host spectra go through pinned memory and a copy kernel, large ones (more
than 1 MiB) through a copy command; device spectra through the copy kernel,
or a copy command where their address is not a multiple of 8 or not device
memory.  Whatever the way, the lists are those of a fresh search, bit for bit.
"""

import time

import numpy as np
import pytest

from fdas_amd import synth
from fdas_amd.host import FDAS

from test_gpu_parity import bank_for, make, spectrum, wide_by_plane

pytestmark = pytest.mark.gpu

H, CAP, T = 4, 64, 5


def lists(f, ab):
    planes, det = wide_by_plane(f, ab, H)
    return [det] + [a for p in planes for a in p]


@pytest.mark.parametrize("n", [1000, 1023, 4999, 1 << 17, (1 << 17) + 1])
def test_every_way_in_gives_the_same_lists(n):
    torch = pytest.importorskip("torch")
    bank = bank_for(T)
    f = make(n, n_templates=T, max_taps=bank.shape[1], tile=1024, n_harmonics=H, cands_per_harmonic=CAP)
    for ab in (FDAS.A, FDAS.B):
        assert f.upload_template_taps(bank, ab), f.last_error
    x, other = spectrum(n, 5), spectrum(n, 6)
    thr = synth.noise_thresholds(x, H)
    loc = np.zeros(f.get_candidate_list_sz(), np.uint32)
    pwr = np.zeros(f.get_candidate_list_sz(), np.float32)

    def searched(ab, start):
        t0 = time.perf_counter()
        assert start() and f.wait(ab), f.last_error
        wall = 1e3 * (time.perf_counter() - t0)
        ms = f.stage_times(ab)
        assert np.all(ms >= 0) and ms[1] > 0 and ms[2] > 0 and ms[3] > 0
        assert ms[:4].sum() <= ms[5] + 1e-3 and ms[5] <= wall
        return lists(f, ab)

    # the FOP itself, once, by the blocking calls
    assert f.perform_input_tiling(x, FDAS.A) and f.perform_ft_convolution(2, FDAS.A), f.last_error
    assert f.perform_harmonic_summing(thr, 2, FDAS.A), f.last_error
    want = lists(f, FDAS.A)
    assert sum(a.size for a in want[1:]) > 0

    def same(got):
        assert all(np.array_equal(a, b) for a, b in zip(got, want))

    same(searched(FDAS.A, lambda: f.launch(x, thr, loc, pwr, 2, FDAS.A)))
    # a second launch of a set that was not waited for: its spectrum, not the first one's
    assert f.launch(other, thr, loc, pwr, 2, FDAS.B), f.last_error
    same(searched(FDAS.B, lambda: f.launch(x, thr, loc, pwr, 2, FDAS.B)))

    raw = torch.zeros(8 * n + 64, dtype=torch.uint8, device="cuda")
    for offset in (0, 8, 4):  # 16-, 8- and 4-byte aligned
        raw.zero_()
        raw[offset:offset + 8 * n] = torch.from_numpy(x.view(np.uint8)).to("cuda")
        torch.cuda.synchronize()
        assert f.set_input_device(raw.data_ptr() + offset, FDAS.B), f.last_error
        same(searched(FDAS.B, lambda: f.launch_resident(thr, loc, pwr, 2, FDAS.B)))
    assert f.launch(other, thr, loc, pwr, 2, FDAS.B) and f.wait(FDAS.B), f.last_error
    pinned = torch.from_numpy(x).pin_memory()
    assert f.set_input_device(pinned.data_ptr(), FDAS.B), f.last_error
    same(searched(FDAS.B, lambda: f.launch_resident(thr, loc, pwr, 2, FDAS.B)))
    f.close()
