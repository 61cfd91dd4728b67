"""Reconstructions whose step puts a point at the foot of an aperture's soft edge: at
1024 x 1024 and 0.35 A one pixel's aperture is 2.0e-7 at (364, 787) and its mirror, less
than the float32 detector centre moves it, and the term there is a unit vector or
nothing.  Held to the object's bar without the undecided points, whose number is held
too; the prepared stack of the same frames by itself."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import OBJ_SCALED, decided_error, engine_for_data, undecided_points

pytestmark = pytest.mark.gpu

ABER = C.MAKE_ENGINE_ABERRATIONS


def _frames(size):
    rng = np.random.default_rng(size)
    data = rng.integers(0, 40, (size, size, 6, 6)).astype(np.uint16)
    data[:, :, 1:5, 1:5] += 300
    return data


@pytest.mark.parametrize("size,step,undecided", [(1024, 0.35, 12), (256, 0.35, 12)])
def test_object_and_prepared_stack(cuda, size, step, undecided):
    data = _frames(size)
    eng = engine_for_data(cuda, data, semiangle_mrad=20.0, det_sampling=9.0, step=step, max_bf=64)
    d = cuda.from_numpy(data).cuda()
    p = O.prepare(data, voltage_kV=300, semiangle_mrad=20.0, det_sampling=9.0, bf_radius=2.0, scan_sampling=step)
    eng.mean_dp(d)
    eng.select_bf(0.0, 2.0)
    eng.prepare_g(d)
    err = np.abs(eng.G_qk.cpu().numpy() - p.G)
    for cols in (slice(0, 1), slice(1, None)):
        assert err[:, :, cols].max() < 2e-6 * np.abs(p.G[:, :, cols]).max()
    points = undecided_points(p.geom, *ABER)
    assert points.sum() <= undecided
    ref = O.object_wave(p.G, p.dc, p.geom, *ABER)
    assert decided_error(eng.reconstruct_object(*ABER).cpu().numpy(), ref, points) < OBJ_SCALED
    obj = cuda.empty((size, size), dtype=cuda.complex64, device="cuda")
    eng.recon_u16(d, *ABER, bf_radius=2.0, obj_out=obj)
    assert decided_error(obj.cpu().numpy(), ref, points) < OBJ_SCALED
