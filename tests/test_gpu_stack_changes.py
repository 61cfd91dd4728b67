"""Handles that outlive a plan's stack: a captured batch of exact losses, replayed
into the same output after the bright field or the stack has changed, gives what
the plain batch gives; a trials handle follows the stack or refuses it."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import engine_for_data, make_engine

pytestmark = pytest.mark.gpu


def _load(eng, torch, num_bf, full=False, seed=0):
    case = C.make_engine_case(128, num_bf)
    half = np.ascontiguousarray(np.roll(case.G, seed, axis=1)[:, :, :65])
    eng.set_bf(case.rows, case.cols, case.center, case.dc)
    eng.import_g(torch.from_numpy(O.expand_hermitian(half) if full else half))
    eng.cache_rotation(0.0)


def _trials(n, odd=False):
    mags, angs = np.zeros((n, 14)), np.full((n, 14), 0.3)
    mags[:, 0] = np.linspace(-150.0, 200.0, n)
    mags[:, 1] = 30.0
    if odd:
        mags[:, 2] = 2.0e3
    return mags, angs, np.linspace(-0.03, 0.04, n)


def test_captured_batch_follows_the_stack(cuda):
    eng = make_engine(cuda, 128, (32, 32), 64, 0.0197, 21.4, (1.0, 1.0), 0.5)
    out = cuda.empty(3, dtype=cuda.float32, device="cuda")
    seen = set()
    for odd in (False, True):
        trials = _trials(3, odd)
        # more pixels, fewer, another stack in the same place, a full plane, and back
        for num_bf, full, seed in [(7, False, 0), (9, False, 0), (60, False, 0), (5, False, 0), (5, False, 3),
                                   (5, True, 0), (7, True, 0), (7, False, 0)]:
            _load(eng, cuda, num_bf, full, seed)
            plain = eng.batch_phase_loss(*trials).cpu().numpy()
            for _ in range(2):
                got = eng.batch_phase_loss(*trials, out=out, graph=True).cpu().numpy()
                np.testing.assert_array_equal(got, plain, err_msg=str((num_bf, full, seed, odd)))
            seen.add(plain.tobytes())
        eng.set_detector_sampling(0.9 / 32.0, 0.9 / 32.0)
        eng.cache_rotation(0.0)
        plain = eng.batch_phase_loss(*trials).cpu().numpy()
        got = eng.batch_phase_loss(*trials, out=out, graph=True).cpu().numpy()
        np.testing.assert_array_equal(got, plain)
        eng.set_detector_sampling(1.0 / 32.0, 1.0 / 32.0)
    assert len(seen) >= 10


def _prepare(eng, d, radius):
    eng.mean_dp(d)
    eng.select_bf(0.0, radius)
    eng.prepare_g(d)
    eng.cache_rotation(0.0)


def _variance(batch, graph):
    return batch.phase_variance(use_graph=graph).cpu().numpy().copy()


@pytest.mark.parametrize("graph", [False, True])
def test_trials_follow_or_refuse_another_stack(cuda, graph):
    """A trials handle takes over a stack of the same size and place, keeps its own
    pixels under a selection that is not prepared, and refuses a stack of another
    size or layout before anything is launched."""
    from quantem.gpu_amd.ssb.compute.hip.trials import TrialBatch
    d, d2 = (cuda.from_numpy(C.poisson_data(s)).cuda() for s in (123, 321))
    eng = engine_for_data(cuda, d, semiangle_mrad=21.4, det_sampling=1.0, step=0.5, max_bf=256)
    trials = _trials(9)

    def fresh():
        batch = TrialBatch([eng], 9)
        batch.set(*trials)
        got = _variance(batch, False)
        batch.close()
        return got

    _prepare(eng, d, 3.2)
    small = TrialBatch([eng], 9)
    small.set(*trials)
    want = _variance(small, graph)
    np.testing.assert_array_equal(want, fresh())
    eng.recon_u16(d2, 0.0, 0.0, 0.0, bf_radius=2.0)           # another selection, the stack untouched
    np.testing.assert_array_equal(_variance(small, graph), want)
    small.set(*trials)
    np.testing.assert_array_equal(_variance(small, graph), want)
    _prepare(eng, d2, 3.2)                                    # another stack in the same place
    want2 = fresh()
    assert not np.array_equal(want2, want)
    np.testing.assert_array_equal(_variance(small, graph), want2)
    eng.set_detector_sampling(1.0 / 18.0, 1.0 / 18.0)
    eng.cache_rotation(0.0)
    np.testing.assert_array_equal(_variance(small, graph), fresh())
    for radius in (4.0, 2.0):                                 # more pixels, fewer
        _prepare(eng, d, radius)
        with pytest.raises(ValueError, match="replaced"):
            small.phase_variance(use_graph=graph)
        with pytest.raises(ValueError, match="replaced"):
            small.set(*trials)
    eng.set_bf([8] * 3, [7, 8, 9], (8.0, 8.0), 1.0)
    eng.import_g(cuda.zeros((3, 128, 65), dtype=cuda.complex64))
    three = TrialBatch([eng], 9)
    three.set(*trials)
    eng.import_g(cuda.zeros((3, 128, 128), dtype=cuda.complex64))
    with pytest.raises(ValueError, match="replaced"):
        three.phase_variance(use_graph=graph)
    eng.plan.close()
    with pytest.raises(ValueError, match="closed"):
        three.phase_variance(use_graph=graph)
    three.close()
    small.close()
