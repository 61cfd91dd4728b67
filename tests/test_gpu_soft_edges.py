"""Overlaps inside an aperture's soft edge under other optics than 20 mrad and coarse
pixels: wide apertures and fine pixels make the edge narrow beside the terms that
cancel in it.  One pixel's stack of unit values gives every point's term; it is held
where the smaller aperture lies strictly inside its edge and |Gamma| > 0.1 A(k).

The bar of 5e-6: a float32 aperture (1.2e-7) moves the direction by 1.2e-6 at most,
the phases of up to 3 half turns by 1.1e-6, sine, cosine and the term by 5e-7, and the
two passes of the object's transform add up to 2e-6 at the worst of the points."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests import _cases as C
from tests._gpu import make_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [128, 256, 512])
@pytest.mark.parametrize("semiangle,ang,voltage", [(20.0, 1.25, 300), (30.0, 0.5, 300), (35.0, 0.35, 200),
                                                   (40.0, 0.25, 300), (60.0, 0.5, 300)])
def test_terms_in_the_soft_edge(cuda, size, semiangle, ang, voltage):
    lam = O.wavelength_angstrom(voltage)
    rout = (semiangle + 0.5 * ang) * 1e-3 / lam
    step = 1.0 / (4.2 * rout)                         # the grid reaches past the lenses
    radius = semiangle / ang
    case = C.make_engine_case(size, 1)
    rng = np.random.default_rng(int(semiangle * 10) + size)
    case.G = np.exp(2j * np.pi * rng.random((1, size, size // 2 + 1))).astype(np.complex64)
    det = min(2 * int(radius) + 8, 256)               # (the largest detector: the disk's middle, at 40 mrad)
    case.det, case.ang_mrad, case.center = (det, det), (ang, ang), (float(det // 2), float(det // 2))
    case.semiangle_mrad, case.wavelength, case.q_step, case.recip, case.dc = semiangle, lam, step, None, 1.0 + 0.0j
    worst = count = 0
    for row, col in ((0.55, 0.2), (-0.3, 0.35), (0.1, -0.72)):
        case.rows = np.array([det // 2 + round(row * radius)], np.int32)
        case.cols = np.array([det // 2 + round(col * radius)], np.int32)
        eng = make_engine(cuda, size, case.det, 1, lam, semiangle, case.ang_mrad, step)
        eng.set_bf(case.rows, case.cols, case.center, case.dc)
        eng.import_g(cuda.from_numpy(case.G))
        eng.cache_rotation(0.0)
        c10 = 1.2 / (lam * rout * rout)
        g = case.geometry()
        got = np.fft.fft2(eng.reconstruct_object(c10, 0.0, 0.0).cpu().numpy().astype(np.complex128))
        ref = O.corrected_fourier_mean(case.G, case.dc, g, c10, 0.0, 0.0)
        qx, qy = g.qx.reshape(-1, 1), g.qy.reshape(1, -1)
        am = O.aperture_geometry(qx - g.kx[0], qy - g.ky[0], g)[3]
        ap = O.aperture_geometry(qx + g.kx[0], qy + g.ky[0], g)[3]
        chi = np.pi * lam * c10 * ((qx * qx) + (qy * qy))
        gamma = np.abs(am * np.exp(-1j * chi) - ap * np.exp(1j * chi))
        low = np.minimum(am, ap)
        held = (low > 1e-3) & (low < 1 - 1e-3) & (gamma > 0.1)
        held[0, 0] = False
        count += int(held.sum())
        worst = max(worst, float(np.abs(got - ref)[held].max(initial=0.0)))
    print(f"{size} {semiangle} mrad {ang} mrad/px {voltage} kV: {worst:.2e} over {count} points")
    assert count > 50
    assert worst < 5e-6
