"""Scan normalisation and the mean diffraction pattern where the frame does not
divide into 16-byte groups: detectors of odd size, smaller than one group,
frames that start off 16 bytes, windows that are cropped on one axis and
padded on the other.  Integers against the oracle bit for bit; the float32
pad frame and mean within one float32 ulp of the float64 sum's (both are
double-float sums rounded once)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import ssb_oracle as O
from tests._gpu import make_engine

pytestmark = pytest.mark.gpu

KINDS = ["uint8", "int8", "uint16", "int16", "uint32", "int32", "float32"]


def _frames(rng, kind, shape):
    if kind == "float32":
        return rng.normal(3.0, 50.0, size=shape).astype(np.float32)
    info = np.iinfo(kind)
    return rng.integers(info.min, info.max, size=shape, dtype=kind, endpoint=True)


def _misaligned(torch, arr):
    """The array on the GPU, one sample past a 16-byte boundary."""
    flat = torch.empty(arr.size + 1, dtype=getattr(torch, str(arr.dtype)), device="cuda")
    view = flat[1:].view(arr.shape)
    view.copy_(torch.from_numpy(arr))
    assert view.is_contiguous() and view.data_ptr() % 16
    return view


def _ulps(a, b):
    return np.abs(a.view(np.int32).astype(np.int64) - b.view(np.int32).astype(np.int64))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("scan,det", [((1, 1), (2, 2)), ((70, 45), (3, 3)), ((128, 127), (5, 7)), ((60, 128), (9, 8)),
                                      ((1030, 40), (2, 3)), ((200, 150), (13, 17))])
def test_normalisation_of_any_frame_size(cuda, kind, scan, det):
    from quantem.gpu_amd.ssb.compute.hip.engine import normalize_scan
    data = _frames(np.random.default_rng(11), kind, scan + det)
    got = normalize_scan(_misaligned(cuda, data)).cpu().numpy()
    ref = O.normalize_scan(data)
    assert got.shape == ref.shape and got.dtype == ref.dtype
    if kind != "float32":
        np.testing.assert_array_equal(got, ref)
        return
    assert _ulps(got, ref).max() <= 1
    T, h, w = ref.shape[0], min(scan[0], ref.shape[0]), min(scan[1], ref.shape[0])
    top, left, r0, c0 = (T - h) // 2, (T - w) // 2, max(0, (scan[0] - T) // 2), max(0, (scan[1] - T) // 2)
    np.testing.assert_array_equal(got[top:top + h, left:left + w], data[r0:r0 + h, c0:c0 + w])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("det", [(1, 1), (2, 2), (3, 3), (5, 7), (8, 8), (61, 83)])
def test_mean_dp_of_any_frame_size(cuda, kind, det):
    data = _frames(np.random.default_rng(12), kind, (128, 128) + det)
    eng = make_engine(cuda, 128, det, 64, O.wavelength_angstrom(300), 21.4, (1.0, 1.0), 0.5)
    sums, mean = eng.mean_dp(_misaligned(cuda, data))
    rs, rm = O.mean_dp(data)
    mean = mean.cpu().numpy()
    if kind == "float32":
        assert _ulps(mean, rm).max() <= 1
    else:
        np.testing.assert_array_equal(sums.cpu().numpy().astype(np.uint64), rs)
        if data.dtype.kind == "u":
            np.testing.assert_array_equal(mean.view(np.uint32), rm.view(np.uint32))
