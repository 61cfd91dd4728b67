"""The network's tiled product and vector kernels at the edges of their tiles:
the tiled bf16 product gives the bits of the general-stride kernel (the same
16-deep products summed in the same order), for every operand layout, partial
tiles, partial K steps and K slices; im2col and its adjoint with and without
whole channel groups against the oracle."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import learned_oracle as L

pytestmark = pytest.mark.gpu


def _operand(torch, x, contiguous_last, pad):
    """``x`` as bf16 bits with its last (or first) axis contiguous in rows
    padded by ``pad``; (tensor, stride of axis 0, stride of axis 1)."""
    y = x if contiguous_last else x.T
    u = (np.asarray(y, np.float32).view(np.uint32) >> 16).astype(np.uint16).view(np.int16)
    buf = np.zeros((y.shape[0], y.shape[1] + pad), np.int16)
    buf[:, :y.shape[1]] = u
    t = torch.tensor(buf, device="cuda")
    ld = buf.shape[1]
    return (t, ld, 1) if contiguous_last else (t, 1, ld)


@pytest.mark.parametrize("ak", [True, False])
@pytest.mark.parametrize("bk", [True, False])
@pytest.mark.parametrize("M,N,K,splits", [(64, 64, 64, 1), (8, 8, 8, 1), (72, 24, 200, 1), (136, 144, 72, 1),
                                          (32, 72, 1096, 4)])
def test_tiled_product_has_the_general_kernels_bits(cuda, ak, bk, M, N, K, splits):
    from quantem.gpu_amd.ssb import learned as Lm
    rng = np.random.default_rng(M * N + K)
    a, b = L.bf16(rng.standard_normal((M, K))), L.bf16(rng.standard_normal((K, N)))
    bias = cuda.tensor(rng.standard_normal(N), dtype=cuda.float32, device="cuda")
    stream = Lm._stream(cuda, cuda.device("cuda", 0))
    got = []
    for pad in (0, 1):                                  # rows of an odd length take the general kernel
        A, sam, sak = _operand(cuda, a, ak, pad)
        B, sbk, sbn = _operand(cuda, b, not bk, pad)
        C = cuda.full((M, N), 3.0, dtype=cuda.float32, device="cuda")
        if splits == 1:
            Lm._call("qnn_gemm_bf16", Lm._p(A), sam, sak, Lm._p(B), sbk, sbn, Lm._p(C), N, 1, Lm._p(bias), M, N, K,
                     1, 1, stream)
        else:
            ws = cuda.empty(splits * M * N, dtype=cuda.float32, device="cuda")
            Lm._call("qnn_gemm_bf16_splitk", Lm._p(A), sam, sak, Lm._p(B), sbk, sbn, Lm._p(C), M, N, K, splits,
                     Lm._p(ws), stream)
        got.append(C.cpu().numpy())
    np.testing.assert_array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    ref = np.maximum(a @ b + bias.cpu().numpy(), 0.0) + 3.0 if splits == 1 else a @ b
    # K products of unit normals in float32: K/2 roundings of 2^-24 of partial sums of size sqrt(K)
    np.testing.assert_allclose(got[0], ref, rtol=0, atol=(K + 2) * 2.0 ** -24 * 4 * np.sqrt(K))


@pytest.mark.parametrize("channels", [3, 4, 8, 16])
def test_im2col_and_adjoint(cuda, channels):
    from quantem.gpu_amd.ssb import learned as Lm
    rng = np.random.default_rng(channels)
    x = rng.standard_normal((3, 6, 4, channels)).astype(np.float32)
    stream = Lm._stream(cuda, cuda.device("cuda", 0))
    X = cuda.tensor(x, device="cuda")
    cols = cuda.empty((3 * 3 * 2, 9 * channels), dtype=cuda.int16, device="cuda")
    Lm._call("qnn_im2col", Lm._p(X), 3, 6, 4, channels, Lm._p(cols), stream)
    bits = cols.cpu().numpy().view(np.uint16).astype(np.uint32) << 16
    np.testing.assert_array_equal(bits.view(np.float32), L.bf16(L.im2col(x)).astype(np.float32))
    d = rng.standard_normal((3 * 3 * 2, 9 * channels)).astype(np.float32)
    D = cuda.tensor(d, device="cuda")
    dX = cuda.empty((3, 6, 4, channels), dtype=cuda.float32, device="cuda")
    Lm._call("qnn_col2im", Lm._p(D), 3, 6, 4, channels, Lm._p(dX), stream)
    ref = L.col2im(d.astype(np.float64), 3, 6, 4, channels)
    np.testing.assert_allclose(dX.cpu().numpy(), ref, rtol=0, atol=4 * 2.0 ** -24 * 16)   # at most 4 terms below 4


def test_one_adam_launch_equals_single_ones(cuda):
    from quantem.gpu_amd.ssb import learned as Lm
    rng = np.random.default_rng(3)
    stream = Lm._stream(cuda, cuda.device("cuda", 0))
    sets = []
    for n in (1, 255, 70000):
        sets.append([cuda.tensor(np.abs(rng.standard_normal(n)), dtype=cuda.float32, device="cuda") for _ in range(4)]
                    + [cuda.zeros(n, dtype=cuda.int16, device="cuda")])
    twins = [[t.clone() for t in s] for s in sets]
    items = [tuple(t.data_ptr() for t in s) + (s[0].numel(),) for s in sets]
    Lm._call("qnn_adam_multi", (Lm._AdamItem * 3)(*items), 3, 1e-3, 0.9, 0.999, 1e-8, 2, stream)
    for s in twins:
        Lm._call("qnn_adam", *(Lm._p(t) for t in s[:4]), s[0].numel(), 1e-3, 0.9, 0.999, 1e-8, 2, Lm._p(s[4]), stream)
    cuda.cuda.synchronize()
    for s, t in zip(sets, twins):
        assert all(cuda.equal(a, b) for a, b in zip(s, t))
    assert Lm._lib().qnn_adam_multi((Lm._AdamItem * 1)(), 17, 1e-3, 0.9, 0.999, 1e-8, 2, ctypes.c_void_p(0)) == -1
