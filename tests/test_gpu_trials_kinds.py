"""The batched search's forms of the overlap, against the FP64 oracle: trials
with C10/C30 only, with C12, with any other even term, with no aberration at
all (the sine of the half sum vanishes everywhere), alone and mixed in one
block of trials; a bright field that reaches past the aperture (pixels with a
zero or partial A(k)); trial counts around a whole block.  The bar is the
search's own: 1e-4 of the variance."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import engine_for_data

pytestmark = pytest.mark.gpu

TERMS = {"none": {}, "radial": {0: 150.0, 4: 9.0e4}, "astig": {0: -90.0, 1: 45.0, 4: -6.0e4},
         "c32": {0: 80.0, 5: 4.0e4}, "c34": {0: -60.0, 6: 5.0e4}, "c50": {0: 120.0, 10: 2.0e7},
         "c52": {1: 30.0, 11: 1.5e7}, "c56": {0: 40.0, 13: 2.0e7}}


def _vectors(kinds):
    mags, angs = np.zeros((len(kinds), 14)), np.zeros((len(kinds), 14))
    for i, k in enumerate(kinds):
        for slot, v in TERMS[k].items():
            mags[i, slot] = v * (1.0 + 0.1 * i)
            angs[i, slot] = 0.4 - 0.05 * i
    return mags, angs, np.radians(np.linspace(-3.0, 4.0, len(kinds)))


@pytest.mark.parametrize("radius", [3.0, 5.0])
@pytest.mark.parametrize("kinds", [["none"], ["radial"] * 8, ["astig"] * 9, list(TERMS),
                                   ["radial"] * 7 + ["c34"] + ["radial"] * 2])
def test_every_form_matches_the_oracle(cuda, kinds, radius):
    from quantem.gpu_amd.ssb.compute.hip.trials import TrialBatch
    data = C.poisson_data(321, radius=6)
    # a semiangle of 3.6 detector pixels: radius 5 takes pixels in and past the soft edge
    eng = engine_for_data(cuda, data, semiangle_mrad=3.6, det_sampling=1.0, step=1.6)
    d = cuda.from_numpy(data).cuda()
    eng.mean_dp(d)
    eng.select_bf(0.0, radius)
    eng.prepare_g(d)
    mags, angs, rot = _vectors(kinds)
    tb = TrialBatch([eng], len(kinds))
    tb.set(mags, angs, rot)
    got = tb.phase_variance(use_graph=False).cpu().numpy()[0].copy()
    p = O.prepare(data, voltage_kV=300, semiangle_mrad=3.6, scan_sampling=1.6, det_sampling=1.0, bf_radius=radius)
    for t in range(len(kinds)):
        geom = O.detector_geometry(p.bf.rows, p.bf.cols, p.bf.center, (16, 16), (1.0, 1.0), p.geom.wavelength, 3.6,
                                   rot[t], 128, 1.6)
        assert got[t] == pytest.approx(O.phase_variance(p.G, p.dc, geom, mags[t], angs[t]), rel=1e-4), kinds[t]
        tb.set(mags[t:t + 1], angs[t:t + 1], rot[t:t + 1])
        assert tb.phase_variance(use_graph=False).cpu().numpy()[0, 0] == got[t], kinds[t]
    tb.close()
