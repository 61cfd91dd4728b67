"""Exact losses over selection sizes around the changes of their split: one pixel, a
split's two, waves of one to four pixels, more pixels than splits and than the
finishing kernel's four-wave form asks for.  The bars are the exact path's own."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import engine_for_case

pytestmark = pytest.mark.gpu

ABER = C.MAKE_ENGINE_ABERRATIONS


@pytest.mark.parametrize("size,num_bf", [(128, n) for n in (1, 2, 3, 31, 33, 65, 130, 257, 300)] +
                         [(256, n) for n in (1, 5, 33, 67)] + [(512, n) for n in (1, 3, 17)] + [(1024, 1), (1024, 5)])
def test_selection_sizes(cuda, size, num_bf):
    full = C.make_engine_case(size, num_bf).G
    case = C.make_engine_case(size, num_bf, g_qk=np.ascontiguousarray(full[:, :, : size // 2 + 1]),
                              bf_center=(15.0, 15.0))
    case.dc = complex(25.0, -8.0) * size
    case.q_step = 0.36
    phase, loss = engine_for_case(cuda, case).reconstruct_with_loss(*ABER)
    ref_phase, ref_loss = O.phase_and_loss(case.G, case.dc, case.geometry(), *ABER)
    assert np.percentile(np.abs(phase.cpu().numpy() - ref_phase), 99.9) < 3e-4
    assert loss == pytest.approx(ref_loss, rel=1e-4, abs=1e-4)
