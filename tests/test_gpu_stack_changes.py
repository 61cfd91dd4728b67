"""Results that outlive a plan's stack: a captured batch of exact losses, replayed
into the same output after the bright field or the stack has changed, gives what
the plain batch gives."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import make_engine

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
