"""ADM map where a wavefront's area is just full, just too small, and too small
from each pair on: lanes of an exact number of bytes, by stretches."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402


def groups(m):
    """A group of 512 elements per entry of m, every lane m bytes of bits: 15
    elements at the center, one 126 k + 1 away with k = 8 (m - 2), above in
    even lanes and below in odd ones (so the center is their mean)."""
    x = np.full((len(m), 32, 16), 32768, np.int64)
    d = 126 * 8 * (np.asarray(m) - 2) + 1
    x[:, 0::2, 5] += d[:, None]
    x[:, 1::2, 5] -= d[:, None]
    return x.reshape(-1).astype(np.uint16)


# 32 groups of a wavefront, 4 waves a ticket, two tickets and a half
@pytest.mark.parametrize("first", [0, 1, 2, 15, 29, 30, 31, 32])
@pytest.mark.parametrize("low,high", [(4, 4), (4, 5), (4, 32), (2, 9), (2, 6), (3, 7)])
def test_area_full_from_each_pair_on(low, high, first):
    # (sums of 32 groups: 128 units of 32 bytes are an area)
    m = np.where(np.arange(320) % 32 >= first, high, low)
    x = groups(m)
    rok, roffs, rcen, rcodes, rbits = oracle.adm_map(x)
    assert rok and rbits.size == 32 * int(m.sum())
    print(f"adm area: {low} then {high} from group {first}", flush=True)
    ws = mans_amd.Workspace(0)
    ok, offs, cen, codes, bits = mans_amd.adm_map(torch.from_numpy(x.view(np.int16)).cuda(), ws)
    assert ok
    assert (offs.cpu().numpy() == roffs).all() and (cen.cpu().numpy().view(np.uint16) == rcen).all()
    assert (codes.cpu().numpy() == rcodes).all() and (bits.cpu().numpy() == rbits).all()
    ws.close()
