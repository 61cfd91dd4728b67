"""Exact losses of stacks far from one: a power of two on the stack and the mean leaves
every phase as it is, bit for bit where nothing overflows or is denormal, also above
2^126, whose reciprocal is denormal.  Below 2^-126 the transforms round to 2^-149: a
mean of 2^-127 leaves 22 bits, 1e-4 of it after the transforms; held to 3e-3."""
from __future__ import annotations

import numpy as np
import pytest

from tests import _cases as C
from tests._gpu import engine_for_case

pytestmark = pytest.mark.gpu

ABER = (150.0, 20.0, 0.3)


def _loss(torch, size, scale, bright):
    rng = np.random.default_rng(size)
    case = C.make_engine_case(size, 5)
    g = rng.integers(-64, 65, (5, size, size // 2 + 1)) + 1j * rng.integers(-64, 65, (5, size, size // 2 + 1))
    case.G = (g * 2.0 ** scale).astype(np.complex64)
    case.dc = 2.0 ** (20 if bright else 10) * 2.0 ** scale
    case.q_step = 0.4
    phase, loss = engine_for_case(torch, case).reconstruct_with_loss(*ABER)
    return phase.cpu().numpy(), loss


@pytest.mark.parametrize("size", [128, 256, 512])
@pytest.mark.parametrize("bright", [True, False])
def test_large_and_small_values(cuda, size, bright):
    want, want_loss = _loss(cuda, size, 0, bright)
    assert np.isfinite(want).all()
    for scale in (-90, 80, 107 if bright else 108):
        phase, loss = _loss(cuda, size, scale, bright)
        np.testing.assert_array_equal(phase, want, err_msg=str(scale))
        assert loss == want_loss
    phase, loss = _loss(cuda, size, -147 if bright else -137, bright)
    assert np.percentile(np.abs(phase - want), 99.9) < 3e-3
    assert loss == pytest.approx(want_loss, rel=3e-3, abs=1e-4)
