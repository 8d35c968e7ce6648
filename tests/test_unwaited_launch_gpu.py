"""GPU test of calls on a buffer set whose launch has not been waited for."""

import time

import numpy as np
import pytest

from fdas_amd import synth
from fdas_amd.host import FDAS

from test_gpu_parity import bank_for, make, spectrum

pytestmark = pytest.mark.gpu

N, T, H, CAP = 20000, 21, 4, 64


@pytest.fixture
def search():
    bank = bank_for(T)
    f = make(N, n_templates=T, max_taps=bank.shape[1], tile=1024, n_harmonics=H, cands_per_harmonic=CAP)
    assert f.upload_template_taps(bank, FDAS.A), f.last_error
    x = spectrum(N, 2)
    yield f, x, synth.noise_thresholds(x, H)
    f.close()


def arrays(f):
    n = f.get_candidate_list_sz()
    return np.zeros(n, np.uint32), np.zeros(n, np.float32)


def test_quantile_thresholds_before_wait_leave_the_launch_its_lists(search):
    """wait() hands over the lists of the launch, also where the quantile thresholds of the set's plane were taken
    between the two; the set's own lists are then the quantile pass's (fewer entries: 3 per plane asked for)."""
    f, x, thr = search
    want = arrays(f)
    assert f.launch(x, thr, *want, 2, FDAS.A) and f.wait(FDAS.A), f.last_error
    assert all((want[1][k * CAP:(k + 1) * CAP] > 0).all() for k in range(H))  # full lists
    q0 = f.quantile_thresholds(3, 2, FDAS.A)
    of_quantile = arrays(f)
    assert f.retrieve_candidates(*of_quantile, FDAS.A)
    assert (of_quantile[1] > 0).sum() < H * CAP
    for again in range(2):
        got = arrays(f)
        assert f.launch_resident(thr, *got, 2, FDAS.A), f.last_error
        for _ in range(1 + again):
            assert np.array_equal(f.quantile_thresholds(3, 2, FDAS.A), q0)
        assert f.wait(FDAS.A), f.last_error
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        after = arrays(f)
        assert f.retrieve_candidates(*after, FDAS.A)
        assert all(np.array_equal(a, b) for a, b in zip(after, of_quantile))
    # a summing pass after it replaces the lists, as it does those of a launch
    got, summed = arrays(f), arrays(f)
    assert f.launch_resident(thr, *got, 2, FDAS.A), f.last_error
    f.quantile_thresholds(3, 2, FDAS.A)
    assert f.perform_harmonic_summing(thr * 2, 2, FDAS.A), f.last_error
    assert f.retrieve_candidates(*summed, FDAS.A) and f.wait(FDAS.A), f.last_error
    assert all(np.array_equal(a, b) for a, b in zip(got, summed))
    assert not np.array_equal(got[0], want[0])


def test_stage_times_of_a_pass_after_an_unwaited_launch(search):
    """The convolution's time stays that of the launch, and the summing's are those of the later pass, though the
    launch's kernels may still be writing theirs when the pass is enqueued."""
    f, x, thr = search
    loc_pwr = arrays(f)
    assert f.launch(x, thr, *loc_pwr, 2, FDAS.A) and f.wait(FDAS.A), f.last_error
    for passes in (lambda: f.perform_harmonic_summing(thr, 2, FDAS.A),
                   lambda: f.quantile_thresholds(3, 2, FDAS.A) is not None,
                   lambda: f.perform_harmonic_summing(thr, 2, FDAS.A) and f.perform_harmonic_summing(thr, 2, FDAS.A)):
        for _ in range(5):
            t0 = time.perf_counter()
            assert f.launch_resident(thr, *loc_pwr, 2, FDAS.A) and passes(), f.last_error
            wall = 1e3 * (time.perf_counter() - t0)
            ms = f.stage_times(FDAS.A)
            assert ms[1] > 0 and ms[2] > 0 and ms[3] > 0, ms
            assert ms[0] + ms[1] + ms[2] + ms[3] <= ms[5] + 1e-3 and ms[5] <= wall, (ms, wall)
            assert f.wait(FDAS.A), f.last_error
    # a launch over an unwaited one: the later one's times
    for again in (lambda: f.launch_resident(thr, *loc_pwr, 2, FDAS.A), lambda: f.launch(x, thr, *loc_pwr, 2, FDAS.A)):
        assert f.launch_resident(thr, *loc_pwr, 2, FDAS.A)
        t0 = time.perf_counter()
        assert again() and f.wait(FDAS.A), f.last_error
        wall = 1e3 * (time.perf_counter() - t0)
        ms = f.stage_times(FDAS.A)
        assert ms[1] > 0 and ms[2] > 0 and ms[3] > 0 and ms[:4].sum() <= ms[5] + 1e-3 and ms[5] <= wall, (ms, wall)


def test_a_launch_over_an_unwaited_one_does_not_wait_for_it(search):
    """Only the copy of the first spectrum has to be over before the second one is staged.  With every bin detected a
    launch's kernels take many times as long as the host needs to enqueue one."""
    f, x, thr = search
    dense = np.zeros(H, np.float32)
    loc_pwr = arrays(f)
    second, device = [], []
    for _ in range(15):
        assert f.launch(x, dense, *loc_pwr, 2, FDAS.A), f.last_error
        t0 = time.perf_counter()
        assert f.launch(x, dense, *loc_pwr, 2, FDAS.A), f.last_error
        second.append(1e3 * (time.perf_counter() - t0))
        f.wait(FDAS.A)  # False: the spill lists overflow
        device.append(f.stage_times(FDAS.A)[5])
    print(f"second launch {np.median(second):.3f} ms on the host, kernels {np.median(device):.3f} ms")
    assert np.median(second) < 0.5 * np.median(device)
    # several in a row: each spectrum was copied before the next took its place
    for seeds in ((3, 4, 2), (2, 3, 4)):
        want, got = arrays(f), arrays(f)
        xs = [spectrum(N, s) for s in seeds]
        assert f.launch(xs[-1], thr, *want, 2, FDAS.A) and f.wait(FDAS.A), f.last_error
        for y in xs:
            assert f.launch(y, thr, *got, 2, FDAS.A), f.last_error
        assert f.wait(FDAS.A) and all(np.array_equal(a, b) for a, b in zip(got, want)), f.last_error
