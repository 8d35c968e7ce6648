"""GPU test of the candidate lists that the selection kernel writes to host memory.

One plan, one served stream and one single-trial context search the same
spectrum again and again while the thresholds change from full lists to fewer
entries to none and back: every pass must equal a fresh search at its
thresholds, bit for bit, so that no entry, kept count or detection count of an
earlier pass is left behind or read too early.
"""

import numpy as np
import pytest

from fdas_amd import synth
from fdas_amd.engine import Engine, Trial
from fdas_amd.host import FDAS

from test_engine_gpu import assert_same, quiet, single_trial
from test_gpu_parity import bank_for, make, spectrum, wide_by_plane

pytestmark = pytest.mark.gpu

CAP = 64
SCALES = (0.8, 1.3, 1e9, 0.8, 1e9, 1.0)  # thresholds: full lists, fewer entries, none, ...


@pytest.fixture(scope="module")
def searched():
    bank = bank_for(85)
    x = spectrum(9001, 77)
    thr = synth.noise_thresholds(x, 8)
    with Engine(tile=2048, cands_per_harmonic=CAP, log=quiet) as eng:
        b = eng.add_bank(bank)
        fresh = {s: eng.run([Trial(x, b, thr * np.float32(s), 2)])[0] for s in set(SCALES)}
    kept = {s: [k.size for k in fresh[s].keys] for s in fresh}
    assert max(kept[0.8]) == CAP and sum(kept[1e9]) == 0
    return bank, x, thr, fresh


@pytest.mark.parametrize("schedule", ["lagged", "streams"])
@pytest.mark.parametrize("graph", [False, True])
def test_plan_passes(searched, schedule, graph):
    bank, x, thr, fresh = searched
    with Engine(tile=2048, cands_per_harmonic=CAP, group_trials=2, groups_in_flight=2, schedule=schedule,
                log=quiet) as eng:
        b = eng.add_bank(bank)
        plan = eng.plan([Trial(x, b, thr, 2) for _ in range(5)], graph=graph)
        for p, s in enumerate(SCALES):
            at = [SCALES[(p + i) % len(SCALES)] for i in range(5)]
            for i in range(5):
                plan.set_trial(i, thresholds=thr * np.float32(at[i]))
            for _ in range(2):
                for i, r in enumerate(plan.run()):
                    assert_same(r, fresh[at[i]])
        plan.close()


def test_served_and_single_passes(searched):
    bank, x, thr, fresh = searched
    with Engine(tile=2048, cands_per_harmonic=CAP, group_trials=3, groups_in_flight=2, log=quiet) as eng:
        b = eng.add_bank(bank)
        for _ in range(3):
            for i, s in enumerate(SCALES):
                eng.submit(Trial(x, b, thr * np.float32(s), 2, tag=i))
            for r in eng.drain():
                assert_same(r, fresh[SCALES[r.tag]])
    f = make(x.size, n_templates=85, max_taps=bank.shape[1], tile=2048, n_harmonics=8, cands_per_harmonic=CAP)
    assert f.upload_template_taps(bank, FDAS.A), f.last_error
    loc = np.zeros(f.get_candidate_list_sz(), np.uint32)
    pwr = np.zeros(f.get_candidate_list_sz(), np.float32)
    for s in SCALES:
        assert f.launch(x, thr * np.float32(s), loc, pwr, 2, FDAS.A), f.last_error
        assert f.wait(FDAS.A), f.last_error
        planes, det = wide_by_plane(f, FDAS.A, 8)
        want, want_det = single_trial(x, bank, thr * np.float32(s), 2, 2048, CAP)
        assert np.array_equal(det, want_det) and np.array_equal(det, fresh[s].n_detected[:8])
        for got, ref in zip(planes, want):
            assert all(np.array_equal(a, r) for a, r in zip(got, ref))
    f.close()
