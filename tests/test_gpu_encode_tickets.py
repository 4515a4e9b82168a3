"""Frames at the encoder's edges, byte for byte against the oracle: input
chunks of 16 bytes a lane, blocks, the units of a wavefront and of a ticket,
and a last block of every kind beside whole ones; inputs only 4-byte
aligned."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# symbols a plane, around: a step, a batch, an input chunk, a block, the
# blocks of a wavefront and a ticket
SIZES = [1, 63, 64, 65, 255, 256, 257, 511, 513, 1023, 1024, 1025, 2049, 4095, 4096, 4097, 8191, 8192, 8193,
         8192 + 4097, 16384 + 511, 8 * 4096 + 1, 8 * 8192 - 1, 8 * 8192, 8 * 8192 + 1, 70000]


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("eb", [1, 2, 4])
def test_frames_at_ticket_edges(lanes, eb):
    import torch

    import mans_amd
    import oracle

    rng = np.random.default_rng(100 * lanes + eb)
    ws = mans_amd.Workspace(0)
    dt = {1: np.uint8, 2: np.uint16, 4: np.uint32}[eb]
    fmt = oracle.FORMAT_NATIVE if lanes == 64 else oracle.FORMAT_REF
    for i, n in enumerate(SIZES):
        p = 9 + i % 3
        v = np.round(rng.laplace(0, float(rng.uniform(0.3, 40)), n)).astype(np.int64)
        x = (v + (1 << (8 * eb - 1))).astype(dt)
        off = 4 // eb * (i % 2)  # every second input starts 4 bytes past a 16-byte boundary
        buf = torch.zeros(n + off, dtype={1: torch.int8, 2: torch.int16, 4: torch.int32}[eb], device="cuda")
        t = buf[off:]
        t.copy_(torch.from_numpy(x.view({1: np.int8, 2: np.int16, 4: np.int32}[eb])))
        out, size = mans_amd.frame_encode(t, mans_amd.params(p, lanes, eb, mans_amd.MODE_PLANES), ws)
        ref = oracle.frame_encode(x, oracle.MODE_PLANES, p, fmt)
        got = out[:size].cpu().numpy()
        assert size == ref.size and (got == ref).all(), (lanes, eb, n, p)
        back = mans_amd.frame_decode(out, size, t.dtype, n, ws)
        assert torch.equal(back, t), (lanes, eb, n, p)
    ws.check()
    ws.close()
