"""The exact loss's two forms against the FP64 oracle: Hermitian stacks under
even aberrations (real transforms, the Nyquist row and columns 0 and N/2 apart)
and the general form beside them (odd aberrations, a full plane).  Random
half-planes, whose columns 0 and N/2 are not Hermitian, with a complex DC above
the modulation (first octants only) and below it (all of them); steps whose
Nyquist row lies inside and outside the apertures; pixels on the axes.  The
bars are the exact path's own (phase p99.9 3e-4, loss 1e-4)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import engine_for_case

pytestmark = pytest.mark.gpu

TERMS = {"none": {}, "radial": {0: 150.0, 4: 9.0e4}, "astig": {0: -90.0, 1: 45.0, 4: -6.0e4},
         "c34": {0: -60.0, 6: 5.0e4}, "coma": {0: 80.0, 2: 3.0e3}}


def _vectors(kind):
    mags, angs = np.zeros(14), np.zeros(14)
    for slot, v in TERMS[kind].items():
        mags[slot], angs[slot] = v, 0.4
    return mags, angs


def _case(size, num_bf, step, bright):
    full = C.make_engine_case(size, num_bf).G
    half = np.ascontiguousarray(full[:, :, : size // 2 + 1])
    case = C.make_engine_case(size, num_bf, g_qk=half, bf_center=(15.0, 15.0))
    case.q_step = step
    case.dc = complex(25.0, -8.0) * size if bright else complex(-0.3, 0.4) * size
    return case


@pytest.mark.parametrize("size,num_bf,step", [(128, 7, 0.5), (128, 130, 0.18), (256, 5, 0.36), (512, 66, 0.5),
                                              (1024, 3, 0.25)])
@pytest.mark.parametrize("bright", [True, False])
def test_forms_match_the_oracle(cuda, size, num_bf, step, bright):
    case = _case(size, num_bf, step, bright)
    eng = engine_for_case(cuda, case)
    for kind in (TERMS if size < 512 else ("astig", "c34")):
        mags, angs = _vectors(kind)
        phase, loss = eng.reconstruct_full_with_loss(mags, angs)
        ref_phase, ref_loss = O.phase_and_loss_full(case.G, case.dc, case.geometry(), mags, angs)
        assert np.percentile(np.abs(phase.cpu().numpy() - ref_phase), 99.9) < 3e-4, kind
        assert loss == pytest.approx(ref_loss, rel=1e-4, abs=1e-4), kind


def test_full_plane_takes_the_general_form(cuda):
    case = _case(128, 7, 0.3, True)
    mags, angs = _vectors("astig")
    half = engine_for_case(cuda, case).reconstruct_full_with_loss(mags, angs)
    full = engine_for_case(cuda, case, O.expand_hermitian(case.G)).reconstruct_full_with_loss(mags, angs)
    assert np.percentile(np.abs((half[0] - full[0]).cpu().numpy()), 99.9) < 3e-4
    assert half[1] == pytest.approx(full[1], rel=1e-4, abs=1e-4)


def test_captured_batches_of_changing_forms(cuda):
    """A captured batch replays with the form its trials need."""
    eng = engine_for_case(cuda, _case(128, 7, 0.4, True))
    out = cuda.empty(3, dtype=cuda.float32, device="cuda")
    rot = np.array([0.0, 0.05, -0.02])
    for kinds in (["none", "astig", "coma"], ["astig", "radial", "coma"], ["c34", "coma", "astig"]):
        mags, angs = (np.stack(v) for v in zip(*map(_vectors, kinds)))
        for scale in (1.0, 0.5, 0.8):
            plain = eng.batch_phase_loss(scale * mags, angs, rot).cpu().numpy()
            got = eng.batch_phase_loss(scale * mags, angs, rot, out=out, graph=True).cpu().numpy()
            np.testing.assert_array_equal(got, plain)


@pytest.mark.parametrize("column", [0, 5, 64])
def test_a_nan_reaches_the_loss(cuda, column):
    case = _case(128, 7, 0.4, True)
    case.G[3, 20, column] = np.nan
    phase, loss = engine_for_case(cuda, case).reconstruct_full_with_loss(*_vectors("astig"))
    assert np.isnan(loss) and bool(phase.isnan().all())
