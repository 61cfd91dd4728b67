"""The decode's search for a block's sequences, on blocks written sequence by
sequence, against the CPU oracle's decoder: sequence counts around one round of
64, the ones that are kept (512) and beyond, length bytes, compressed sizes
around the staging buffer's at every alignment, chunks in one buffer; and every
kind of malformed sequence, refused with the frames around it intact.  Integers:
equal."""
from __future__ import annotations

import struct

import numpy as np
import pytest

from oracle import bslz4_oracle as B

pytestmark = pytest.mark.gpu

BLOCK = 8192


def _length(extra):
    out = b""
    while extra >= 255:
        out, extra = out + b"\xff", extra - 255
    return out + bytes([extra])


def _seq(lit, off=None, ml=0):
    """One LZ4 sequence: literals, then a match of ml >= 4 bytes (off None: none)."""
    m = ml - 4
    out = bytes([(min(len(lit), 15) << 4) | (min(m, 15) if off is not None else 0)])
    out += (_length(len(lit) - 15) if len(lit) >= 15 else b"") + lit
    if off is not None:
        out += struct.pack("<H", off) + (_length(m - 15) if m >= 15 else b"")
    return out


def _chunk(payloads):
    body = b"".join(struct.pack(">I", len(p)) + p for p in payloads)
    return struct.pack(">QI", BLOCK * len(payloads), BLOCK) + body


def _fill(rng, n_seq, literals):
    """A block of n_seq sequences, about `literals` literal bytes in all."""
    seqs, size = [], 0
    for i in range(n_seq - 2):
        lit = rng.integers(0, 256, max(int(i == 0), literals // n_seq)).astype(np.uint8).tobytes()
        ml = int(rng.integers(4, 7))
        off = int(rng.integers(1, size + len(lit) + 1))
        seqs.append(_seq(lit, off, ml))
        size += len(lit) + ml
    tail = rng.integers(0, 256, 9).astype(np.uint8).tobytes()
    pad = rng.integers(0, 256, max(1 if size == 0 else 0, literals % n_seq)).astype(np.uint8).tobytes()
    seqs.append(_seq(pad, 1, BLOCK - size - len(pad) - 9))
    return b"".join(seqs) + _seq(tail)


def _expect(payload):
    return B.bitunshuffle(B.lz4_decompress(payload, BLOCK), BLOCK // 2, np.uint16)


@pytest.mark.parametrize("n_seq", [2, 3, 63, 64, 65, 128, 129, 400, 511, 512, 513, 640])
def test_sequence_counts(cuda, n_seq):
    from quantem.gpu_amd.ssb.compute.hip.bslz4 import decode_u16
    rng = np.random.default_rng(n_seq)
    blocks = [_fill(rng, n_seq, 40), _fill(rng, max(2, n_seq // 2), 300), _fill(rng, n_seq, 0)]
    out = decode_u16([_chunk([b]) for b in blocks], (1, 64, 64)).cpu().numpy()
    for got, b in zip(out, blocks):
        np.testing.assert_array_equal(got.ravel(), np.asarray(_expect(b)).ravel())


@pytest.mark.parametrize("size", [2040, 2044, 2045, 2046, 2047, 2048, 2049, 2300])
def test_sizes_around_the_staging_buffer(cuda, size):
    """Literal runs that make the compressed block `size` bytes, after chunks
    that shift it to every alignment."""
    from quantem.gpu_amd.ssb.compute.hip.bslz4 import decode_u16
    rng = np.random.default_rng(size)
    blocks = []
    for shift in range(4):
        blocks.append(_fill(rng, 5, 20 + shift))
        lit = size - 80
        while True:
            body = rng.integers(0, 256, lit).astype(np.uint8).tobytes()
            b = _seq(body, 7, 300) + _seq(b"", 1, BLOCK - lit - 309) + _seq(body[:9])
            if len(b) >= size:
                break
            lit += size - len(b)
        blocks.append(b)
    out = decode_u16([_chunk([b]) for b in blocks], (1, 64, 64)).cpu().numpy()
    for got, b in zip(out, blocks):
        np.testing.assert_array_equal(got.ravel(), np.asarray(_expect(b)).ravel())


GOOD = _seq(b"abcdefgh", 3, 20)
END = _seq(b"012345678")
MALFORMED = {
    "offset 0": GOOD + _seq(b"x", 0, BLOCK - 38) + END,
    "offset before the start": _seq(b"abc", 4, BLOCK - 12) + END,
    "match past the block": GOOD + _seq(b"x", 2, BLOCK) + END,
    "literals past the block": GOOD + _seq(bytes(2000), 1, BLOCK - 1900) + END,
    "literals past the stream": GOOD + bytes([0xF0, 200]) + b"short",
    "length bytes past the stream": GOOD + bytes([0xF0]) + b"\xff" * 20,
    "an endless length": GOOD + bytes([0x1F]) + b"z" + b"\x01\x00" + b"\xff" * 60 + b"\x01" + END,
    "ends with a match": GOOD + _seq(b"x", 1, BLOCK - 29),
    "offset cut off": GOOD + bytes([0x10]) + b"x\x01",
    "block too short": GOOD + _seq(b"x", 1, 4000) + END,
    "empty": b"",
    "late": _fill(np.random.default_rng(1), 200, 40)[:-3],
}


@pytest.mark.parametrize("kind", list(MALFORMED))
def test_malformed_sequences_are_refused(cuda, kind):
    from quantem.gpu_amd.ssb.compute.hip.bslz4 import decode_u16
    good = _fill(np.random.default_rng(5), 70, 100)
    with pytest.raises(ValueError, match="malformed"):
        decode_u16([_chunk([good]), _chunk([MALFORMED[kind]]), _chunk([good])], (1, 64, 64))
    out = decode_u16([_chunk([good])], (1, 64, 64)).cpu().numpy()
    np.testing.assert_array_equal(out.ravel(), np.asarray(_expect(good)).ravel())


def test_a_large_buffer_is_parsed_ahead(cuda):
    """Beyond 48 MiB of compressed bytes the sequences come from the parse: the
    same frames, and a malformed block still refused."""
    from quantem.gpu_amd.ssb.compute.hip.bslz4 import Bslz4Chunks
    rng = np.random.default_rng(9)
    kinds = [_chunk([_fill(rng, n, lit)]) for n, lit in ((2, 0), (64, 40), (65, 900), (300, 100), (640, 0))]
    kinds.append(_chunk([_seq(rng.integers(0, 256, 6000).astype(np.uint8).tobytes(), 5, BLOCK - 6009) + END]))
    order = np.concatenate([np.arange(6), rng.integers(4, 6, 17000)])
    buf = np.frombuffer(b"".join(kinds[i] for i in order), dtype=np.uint8).copy()
    sizes = np.array([len(kinds[i]) for i in order], dtype=np.int64)
    assert buf.size > 48 << 20
    want = [np.asarray(_expect(k[16:])).reshape(64, 64) for k in kinds]
    out = Bslz4Chunks((buf, sizes), (1, 64, 64)).decode().cpu().numpy()
    for i in list(range(40)) + list(range(len(order) - 40, len(order))):
        np.testing.assert_array_equal(out[i], want[order[i]])
    for k in range(6):
        ids = np.flatnonzero(order == k)
        assert (out[ids].astype(np.int64).sum(axis=(1, 2)) == want[k].astype(np.int64).sum()).all()
    bad = buf.copy()
    bad[16 + 2:16 + 4] = 0xFF                                        # the first block's offset
    with pytest.raises(ValueError, match="malformed"):
        Bslz4Chunks((bad, sizes), (1, 64, 64)).decode()
