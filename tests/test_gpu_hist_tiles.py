"""The histogram launch (matrix-core tiles of 4 KiB, single bytes around
them) against numpy.bincount: sizes around the tiles, chunks and wavefront
rounds, unaligned starts, and bytes at the extremes of the float sums (every
nibble at its largest value, a few smallest terms among them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 15, 17, 4095, 4096, 4097, 8 * 4096 - 1, 8 * 4096 + 1, 16 * 4096 + 5, 40 * 4096 + 3, 1 << 20, 5_000_011]


@pytest.mark.parametrize("stride", [1, 2, 4])
@pytest.mark.parametrize("kind", ["random", "largest", "largest_and_smallest", "skewed"])
def test_histogram_tiles(stride, kind):
    import torch

    import mans_amd

    rng = np.random.default_rng(stride)
    ws = mans_amd.Workspace(0)
    for n in SIZES:
        if kind == "random":
            x = rng.integers(0, 256, n + 16, dtype=np.uint8)
        elif kind == "largest":
            x = np.full(n + 16, 0x77, np.uint8)
        elif kind == "largest_and_smallest":
            x = np.where(rng.random(n + 16) < 1e-3, 0x11, 0xf7).astype(np.uint8)
        else:
            x = np.minimum(rng.geometric(0.4, n + 16) + 120, 255).astype(np.uint8)
        t = torch.from_numpy(x).cuda()
        for off in (0, 4, 12):
            m = n // stride * stride
            got = mans_amd.histogram(t[off:off + m], ws, stride=stride).cpu().numpy()
            ref = np.bincount(x[off:off + m:stride], minlength=256)
            assert (got == ref).all(), (kind, stride, n, off)
    ws.close()
