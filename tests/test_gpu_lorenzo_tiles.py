"""The Lorenzo inverse by tiles (4, 8 or 16 planes by 8 to 32 rows by whole
rows of up to eight chunks of 1024) at the edges of the tiles, against 32-bit
prefix sums; and the other route, taken where buffers overlap or the tiles do
not fit a launch, which must give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

EB = 0.25
SHAPES = [(1, 1, 1), (1, 1, 63), (1, 9, 64), (2, 1, 65), (16, 8, 1024), (17, 9, 1023), (33, 33, 100), (15, 31, 1025),
          (9, 17, 2048), (8, 40, 2049), (5, 33, 4096), (4, 9, 4097), (3, 10, 8192), (100, 300, 130), (300, 64, 20),
          (16 * 65535 + 1, 1, 1), (16 * 65535, 1, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_inverse_is_the_prefix_sum(shape):
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    r = rng.integers(-500, 501, n).astype(np.int64)
    idx = np.flatnonzero(rng.random(n) < 0.01).astype(np.uint32)
    r[idx] = rng.integers(-(1 << 30), 1 << 30, idx.size)
    codes = (32768 + r).astype(np.uint16)
    codes[idx] = 0
    q = r.reshape(shape)
    for axis in range(3):
        q = np.cumsum(q, axis=axis)
    want = q.astype(np.uint64).astype(np.uint32).view(np.int32).astype(np.float32) * np.float32(2 * EB)
    print(f"lorenzo inverse {shape} outliers {idx.size}", flush=True)
    perm = rng.permutation(idx.size)
    ti = torch.from_numpy(idx[perm].view(np.int32)).cuda()
    tv = torch.from_numpy(r[idx][perm].astype(np.int32)).cuda()
    tc = torch.from_numpy(codes.view(np.int16)).cuda()
    ws = mans_amd.Workspace(0)
    got = mans_amd.lorenzo_reconstruct(tc, ti, tv, shape, EB, ws)
    ws.check()
    assert (got.cpu().numpy().view(np.uint32) == want.view(np.uint32)).all()
    # codes in the field's own memory
    buf = torch.zeros(n, dtype=torch.float32, device="cuda")
    inside = buf.view(torch.int16)[n:2 * n] if n > 1 else buf.view(torch.int16)[:1]
    inside.copy_(tc)
    again = mans_amd.lorenzo_reconstruct(inside, ti, tv, shape, EB, ws, out=buf.view(shape))
    ws.check()
    assert torch.equal(again.view(torch.int32), got.view(torch.int32))
    ws.close()
