"""Batched decode at the edges of its work items: a workgroup takes up to 4 or
16 tickets of a buffer (a ticket: two blocks of a uint8 buffer, one block's
plane pair of wider elements; a uint32 buffer's second pair starts an item of
its own), and the LUTs of the item before must not be read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

DT = {1: np.uint8, 2: np.uint16, 4: np.uint32}
VIEW = {1: np.uint8, 2: np.int16, 4: np.int32}


@pytest.mark.parametrize("run", [0, 1, 4])
@pytest.mark.parametrize("p,lanes", [(9, 64), (10, 64), (11, 64), (10, 32)])
@pytest.mark.parametrize("eb", [1, 2, 4])
def test_items_of_every_size(eb, p, lanes, run):
    block = 128 * lanes
    per = 2 if eb == 1 else 1  # blocks per ticket
    sizes = [0, 1, 0]
    for tickets in (1, 3, 4, 5, 15, 16, 17, 33):
        sizes += [tickets * per * block - 1, tickets * per * block, (tickets * per - 1) * block + 1]
    rng = np.random.default_rng(eb * 100 + p * 10 + lanes + run)
    xs = [np.round(rng.laplace(0, 0.5 + 3 * (i % 7), n)).astype(np.int64).astype(DT[eb]) for i, n in enumerate(sizes)]
    print(f"eb {eb} p {p} lanes {lanes} run {run} buffers {len(xs)}", flush=True)
    like = [torch.from_numpy(x.view(VIEW[eb])).cuda() for x in xs]
    ws = mans_amd.Workspace(0)
    q = mans_amd.params(p, lanes, eb, mans_amd.MODE_PLANES)
    frames = []
    for t in like:
        f, size = mans_amd.frame_encode(t, q, ws)
        frames.append(f[:size].clone())
    mans_amd.set_batch_grain(0, 0, run)
    try:
        dec = mans_amd.DecodeBatch(frames, [f.numel() for f in frames], like, mans_amd.params(p, lanes), ws)
        for _ in range(3):
            got = dec.run()
            torch.cuda.synchronize()
            ws.check()
            for i, x in enumerate(xs):
                assert (got[i].cpu().numpy().view(x.dtype) == x).all(), (i, x.size)
                got[i].zero_()
        dec.close()
    finally:
        mans_amd.set_batch_grain(0, 0, 0)
        ws.close()
