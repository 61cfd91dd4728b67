"""Plan buffers lent by torch's caching allocator: given back when the plan
closes, ordered behind the work that last used them on a side stream, and safe
for sessions that start and end in several threads.  Every result is the same
bits as the first one."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from tests import _cases as C
from tests._gpu import engine_for_data

pytestmark = pytest.mark.gpu


def _session(torch, d):
    eng = engine_for_data(torch, d, semiangle_mrad=21.4, det_sampling=1.0, step=0.5, max_bf=256)
    eng.mean_dp(d)
    eng.select_bf(0.0, 3.0)
    eng.prepare_g(d)
    eng.cache_rotation(0.0)
    phase, loss = eng.reconstruct_with_loss(*C.MAKE_ENGINE_ABERRATIONS)
    out = phase.cpu().numpy(), loss
    eng.plan.close()
    return out


def test_closing_gives_the_memory_back(cuda):
    d = cuda.from_numpy(C.poisson_data(123)).cuda()
    _session(cuda, d)
    before = cuda.cuda.memory_allocated()
    _session(cuda, d)
    assert cuda.cuda.memory_allocated() == before


def test_side_streams_and_threads(cuda):
    d = cuda.from_numpy(C.poisson_data(123)).cuda()
    want = _session(cuda, d)
    cuda.cuda.synchronize()
    got = {}

    def work(i):
        with cuda.cuda.stream(cuda.cuda.Stream()):
            for _ in range(3):
                # blocks go back with writes to them still queued on this stream
                junk = [cuda.empty(1 << 25, dtype=cuda.float32, device="cuda").fill_(float("nan")) for _ in range(4)]
                del junk
                got[i] = _session(cuda, d)
                if not np.array_equal(got[i][0], want[0]) or got[i][1] != want[1]:
                    return

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 3
    for phase, loss in got.values():
        np.testing.assert_array_equal(phase, want[0])
        assert loss == want[1]
