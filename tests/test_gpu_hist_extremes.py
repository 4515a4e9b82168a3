"""The matrix-core histogram where its float and integer sums are largest:
bytes whose terms are all the largest (or nearly all, with a few of the
smallest), for as many tiles as an accumulator ever holds; inputs of more
chunks than the grid; and inputs so long that a wavefront empties its integer
sums in between."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

# both nibbles 7: every term of a row and column 36; 0xf7 / 0x7f: of both signs
KINDS = {"largest": [(0x77, 1)], "largest_and_smallest": [(0x77, 1), (0x11, 1009)],
         "signs": [(0xf7, 1), (0x7f, 3), (0x88, 1013)], "other": [(0xff, 1), (0x00, 5), (0x70, 1021)]}


def fill(n, kind):
    """n bytes: the kind's first value, the others at every step-th byte."""
    x = torch.empty(n, dtype=torch.uint8, device="cuda")
    for value, step in KINDS[kind]:
        x[::step] = value
    return x


def counts(x, stride):
    """Counts of the bytes at the elements' first position."""
    out = torch.zeros(256, dtype=torch.int64)
    left = x.numel() // stride
    for value in sorted({v for k in KINDS.values() for v, _ in k}):
        for i in range(0, x.numel(), 1 << 30):
            out[value] += int((x[i:i + (1 << 30)][::stride] == value).sum())
        left -= int(out[value])
    assert left == 0
    return out.numpy()


@pytest.mark.parametrize("stride", [1, 2, 4])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_more_chunks_than_the_grid(kind, stride):
    ws = mans_amd.Workspace(0)
    x = fill((96 << 20) + 20, kind)
    got = mans_amd.histogram(x, ws, stride=stride).cpu().numpy().view(np.uint32)
    assert (got == counts(x, stride)).all()
    ws.close()


@pytest.mark.parametrize("stride", [2, 4])
def test_sums_emptied_in_between(stride):
    # 512 workgroups of 8 wavefronts, 256 tiles of 4 KiB each before a flush:
    # 4 GiB, and half as much again
    ws = mans_amd.Workspace(0)
    x = fill(6 << 30, "largest_and_smallest")
    print(f"histogram of 6 GiB, stride {stride}", flush=True)
    got = mans_amd.histogram(x, ws, stride=stride).cpu().numpy().view(np.uint32)
    assert (got == counts(x, stride)).all()
    ws.close()


@pytest.mark.parametrize("eb", [1, 2, 4])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_batched_chunks_of_the_largest_grain(kind, eb):
    # a wavefront counts 32 tiles of a 512 KiB chunk, 16 in float at a time
    n = (5 << 20) // eb + 3
    x = fill(n * eb, kind).view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[eb])
    ws = mans_amd.Workspace(0)
    mans_amd.set_batch_grain(1 << 19, 0, 0)
    try:
        b = mans_amd.EncodeBatch([x], mans_amd.params(10, 64), ws)
        size = int(b.run()[0])
        ws.check()
    finally:
        mans_amd.set_batch_grain(0, 0, 0)
    ref = oracle.frame_encode(x.cpu().numpy().view({1: np.uint8, 2: np.uint16, 4: np.uint32}[eb]),
                              oracle.MODE_PLANES, 10, oracle.FORMAT_NATIVE)
    assert size == ref.size and (b.outs[0][:size].cpu().numpy() == ref).all()
    b.close()
    ws.close()
