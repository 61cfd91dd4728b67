"""Aberrations under which Gamma vanishes or nearly does, against the FP64 oracle:
none, tiny ones (2 A(k) |sin(pi s)| below, at and above the guard of 1e-8), and
C12 alone or as large as C10, which cancel on the diagonals or on an axis.  Every
path: the object of a resident stack, reconstructions, the exact loss and the
batched search.  The bars are the paths' own; the search's variance of a phase
that vanishes is held to 1e-10, a phase error of 1e-5."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import (OBJ_SCALED, decided_error, engine_for_case, engine_for_data, scaled_error,
                        undecided_points)

pytestmark = pytest.mark.gpu

SMALL = [(0.0, 0.0, 0.0), (1e-9, 0.0, 0.0), (1e-7, 0.0, 0.0), (-1e-5, 0.0, 0.0), (0.0, 1e-14, 0.0)]
CANCELLING = [(0.0, 5.0, 0.0), (0.0, 30.0, 0.0), (25.0, 25.0, 0.0)]
ALL = SMALL + CANCELLING


def _case(size, num_bf, step):
    full = C.make_engine_case(size, num_bf).G
    half = np.ascontiguousarray(full[:, :, : size // 2 + 1])
    case = C.make_engine_case(size, num_bf, g_qk=half, bf_center=(15.0, 15.0))
    case.q_step = step
    return case


@pytest.mark.parametrize("size,num_bf,step,aberrations", [(128, 7, 0.4, ALL), (256, 7, 0.4, ALL),
                                                          (512, 3, 0.4, [SMALL[2], CANCELLING[1]]),
                                                          (1024, 2, 0.5, [SMALL[3], CANCELLING[0]])])
def test_object(cuda, size, num_bf, step, aberrations):
    case = _case(size, num_bf, step)
    eng = engine_for_case(cuda, case)
    for aber in aberrations:
        obj = eng.reconstruct_object(*aber).cpu().numpy()
        assert scaled_error(obj, O.object_wave(case.G, case.dc, case.geometry(), *aber)) < OBJ_SCALED, aber


@pytest.mark.parametrize("size,step,aberrations", [(128, 0.9, ALL), (256, 0.9, ALL),
                                                   (512, 0.9, [SMALL[2], CANCELLING[1]]),
                                                   (1024, 0.9, [SMALL[3]])])
def test_reconstruction(cuda, size, step, aberrations):
    """From frames, and the prepared stack's object the same.  The detector's
    centre, which the frames give, puts some points on the diagonals where both
    apertures differ by 1e-7 only, beside a sine that is no larger."""
    rng = np.random.default_rng(size)
    data = rng.integers(0, 40, (size, size, 6, 6)).astype(np.uint16)
    data[:, :, 1:5, 1:5] += 300
    eng = engine_for_data(cuda, data, semiangle_mrad=20.0, det_sampling=9.0, step=step, max_bf=64)
    d = cuda.from_numpy(data).cuda()
    p = O.prepare(data, scan_sampling=step, voltage_kV=300, semiangle_mrad=20.0, det_sampling=9.0, bf_radius=2.0)
    objs = []
    for aber in aberrations:
        obj = cuda.empty((size, size), dtype=cuda.complex64, device="cuda")
        eng.recon_u16(d, *aber, bf_radius=2.0, obj_out=obj)
        objs.append(obj.cpu().numpy())
        undecided = undecided_points(p.geom, *aber)
        assert undecided.mean() < 2e-3
        assert decided_error(objs[-1], O.object_wave(p.G, p.dc, p.geom, *aber), undecided) < OBJ_SCALED, aber
    eng.mean_dp(d)
    eng.select_bf(0.0, 2.0)
    eng.prepare_g(d)
    for aber, obj in zip(aberrations, objs):
        assert scaled_error(eng.reconstruct_object(*aber).cpu().numpy(), obj) < OBJ_SCALED, aber


@pytest.mark.parametrize("size,num_bf,step,aberrations", [(128, 7, 0.4, ALL), (256, 5, 0.36, [SMALL[1], *CANCELLING]),
                                                          (512, 3, 0.4, [SMALL[2], CANCELLING[1]])])
def test_loss(cuda, size, num_bf, step, aberrations):
    case = _case(size, num_bf, step)
    case.dc = complex(25.0, -8.0) * size
    eng = engine_for_case(cuda, case)
    for aber in aberrations:
        phase, loss = eng.reconstruct_with_loss(*aber)
        ref_phase, ref_loss = O.phase_and_loss(case.G, case.dc, case.geometry(), *aber)
        assert np.percentile(np.abs(phase.cpu().numpy() - ref_phase), 99.9) < 3e-4, aber
        assert loss == pytest.approx(ref_loss, rel=1e-4, abs=1e-4), aber


def test_search(cuda):
    from quantem.gpu_amd.ssb.compute.hip.trials import TrialBatch
    data = C.poisson_data(321, radius=6)
    eng = engine_for_data(cuda, data, semiangle_mrad=3.6, det_sampling=1.0, step=1.6)
    d = cuda.from_numpy(data).cuda()
    eng.mean_dp(d)
    eng.select_bf(0.0, 5.0)
    eng.prepare_g(d)
    p = O.prepare(data, voltage_kV=300, semiangle_mrad=3.6, scan_sampling=1.6, det_sampling=1.0, bf_radius=5.0)
    mags, angs = np.zeros((len(ALL), 14)), np.zeros((len(ALL), 14))
    for i, (c10, c12, _) in enumerate(ALL):
        mags[i, :2] = c10, c12
    tb = TrialBatch([eng], len(ALL))
    tb.set(mags, angs)
    got = tb.phase_variance(use_graph=False).cpu().numpy()[0]
    for i, aber in enumerate(ALL):
        assert got[i] == pytest.approx(O.phase_variance(p.G, p.dc, p.geom, mags[i], angs[i]), rel=1e-4, abs=1e-10), aber
    tb.close()
