"""CPU model of the encoder's table entry (mans_amd/csrc/codec_device.hpp,
enc_entry / enc_quot / enc_next): the quotient taken from it is exact for
every frequency, and so are the emission test, the renormalised quotient and
the next state that follow from it."""
import numpy as np
import pytest


def entry(pdf: int, cdf: int, p: int) -> tuple[int, int]:
    s = (pdf - 1).bit_length()
    magic = ((1 << 32) * ((1 << s) - pdf)) // pdf + 1  # the normaliser's
    x = (((1 << p) - pdf) << 16) | (cdf << 5) | s
    y = 0x80000000 + (magic >> 1) + (magic & 1)
    return x, y


@pytest.mark.parametrize("p", [9, 10, 11])
def test_entry_gives_exact_quotients_and_states(p):
    rng = np.random.default_rng(p)
    W = 1 << p
    for pdf in range(1, W + 1):
        cdf = int(rng.integers(0, W - pdf + 1))
        ex, ey = entry(pdf, cdf, p)
        assert ex < 1 << 32 and 1 << 31 <= ey < 1 << 32
        # states at the edges of every kind of step, multiples of pdf and
        # their neighbours, and random ones
        k = rng.integers(0, (1 << 31) // pdf, 64, dtype=np.uint64) * np.uint64(pdf)
        thr = pdf << (31 - p)
        x = np.concatenate([k, k + np.uint64(pdf - 1), k + np.uint64(1),
                            np.array([1 << 15, (1 << 31) - 1, thr - 1, thr, thr + 1, (1 << 16) * pdf,
                                      (1 << 16) * pdf - 1], np.uint64),
                            rng.integers(1 << 15, 1 << 31, 64, dtype=np.uint64)])
        x = x[(x >= 1 << 15) & (x < 1 << 31)]
        q = (((x + x) * np.uint64(ey)) >> np.uint64(32)) >> np.uint64(ex & 31)
        assert (q == x // np.uint64(pdf)).all(), (p, pdf)
        emit = q >= 1 << (31 - p)
        assert (emit == (x >= thr)).all()
        xr = np.where(emit, x >> np.uint64(16), x)
        qr = np.where(emit, q >> np.uint64(16), q)
        assert (qr == xr // np.uint64(pdf)).all() and (qr < 1 << 24).all()
        nxt = qr * np.uint64(ex >> 16) + xr + np.uint64((ex >> 5) & 0x7ff)
        ref = (xr // np.uint64(pdf)) * np.uint64(W) + xr % np.uint64(pdf) + np.uint64(cdf)
        assert (nxt == ref).all() and (nxt < 1 << 31).all()
