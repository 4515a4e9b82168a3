"""The Lorenzo inverse by tiles of every height (the rows of a tile grow and
shrink with the field's shape), with a last band and slab cut off, bit for bit
against 64-bit prefix sums; and a workspace frozen by a captured call serves a
field of any shape with as many elements."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402
from test_lorenzo_inverse_plan import plan  # noqa: E402

EB = 0.25


def field(shape, seed):
    """Codes, outlier indices and residuals of a random field, and the field."""
    n = shape[0] * shape[1] * shape[2]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = torch.randint(-500, 501, (n,), generator=g, device="cuda", dtype=torch.int64)
    idx = torch.nonzero(torch.rand(n, generator=g, device="cuda") < 1e-3).reshape(-1)
    r[idx] = torch.randint(-(1 << 30), 1 << 30, (idx.numel(),), generator=g, device="cuda", dtype=torch.int64)
    codes = 32768 + r
    codes[idx] = 0
    codes = torch.where(codes >= 32768, codes - 65536, codes).to(torch.int16)
    val = r[idx].to(torch.int32)
    q = r.reshape(shape)
    for dim in range(3):
        q = torch.cumsum(q, dim)
    q = ((q + (1 << 31)) % (1 << 32)) - (1 << 31)  # 32-bit sums wrap
    return codes, idx.to(torch.int32), val, q.to(torch.float32) * (2 * EB)


# shape, and the rows of a tile on 256 compute units
SHAPES = [((64, 64, 64), 2), ((128, 130, 400), 4), ((130, 500, 66), 8), ((500, 499, 70), 16), ((700, 330, 400), 32),
          ((100, 330, 1030), 8), ((200, 301, 1500), 32), ((60, 90, 2050), 8), ((100, 333, 2050), 8),
          ((24, 130, 4100), 4), ((64, 90, 4100), 8), ((1, 200_001, 7), 64), ((33, 200_003, 5), 64),
          ((1, 600_001, 3), 256)]


@pytest.mark.parametrize("shape,rows", SHAPES, ids=lambda v: str(v).replace(" ", ""))
def test_inverse_at_every_tile_height(shape, rows):
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    print(f"lorenzo inverse {shape} rows {plan(*shape, cu).ty}", flush=True)
    if cu == 256:
        assert plan(*shape, cu).ty == rows
    codes, idx, val, want = field(shape, sum(shape))
    ws = mans_amd.Workspace(0)
    got = mans_amd.lorenzo_reconstruct(codes, idx, val, shape, EB, ws)
    ws.check()
    assert torch.equal(got.view(torch.int32).reshape(-1), want.view(torch.int32).reshape(-1))
    ws.close()


def test_frozen_workspace_serves_any_shape_of_its_size():
    # 4 bytes an element, from a call whose field overlaps its codes; frozen
    # by a capture of the same call
    n = 500_000
    ws = mans_amd.Workspace(0)
    buf = torch.zeros(n, dtype=torch.float32, device="cuda")
    none = torch.zeros(0, dtype=torch.int32, device="cuda")
    inside = buf.view(torch.int16)[n:]
    inside.fill_(-32768)
    mans_amd.lorenzo_reconstruct(inside, none, none, (5, 100, 1000), EB, ws, out=buf.view(5, 100, 1000))
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        mans_amd.lorenzo_reconstruct(inside, none, none, (5, 100, 1000), EB, ws, out=buf.view(5, 100, 1000), stream=s)
    for shape in ((1, 500, 1000), (5, 100, 1000), (1, 100, 5000), (5, 20, 5000), (250, 2000, 1), (1, 500_000, 1)):
        codes, idx, val, want = field(shape, sum(shape))
        got = mans_amd.lorenzo_reconstruct(codes, idx, val, shape, EB, ws)
        ws.check()
        assert torch.equal(got.view(torch.int32).reshape(-1), want.view(torch.int32).reshape(-1)), shape
    del graph
    ws.close()


# rows over 2048: tiles of 4 planes and 2 rows.  Tiles an axis of 1, 2 (no
# prefixes), 3, and 8 and 9 slabs (a tile sums its corners, or a launch does)
@pytest.mark.parametrize("shape", [(4, 2, 3000), (4, 4, 3000), (8, 2, 3000), (8, 4, 3000), (7, 3, 2049), (9, 6, 3000),
                                   (5, 5, 8192), (32, 6, 2500), (30, 5, 2500), (36, 6, 2500), (33, 3, 2051),
                                   (36, 1, 2500), (1, 6, 2500), (130, 70, 33), (113, 61, 200)],
                         ids=lambda v: "x".join(map(str, v)))
def test_inverse_of_few_tiles(shape):
    assert plan(*shape).fits
    codes, idx, val, want = field(shape, sum(shape))
    ws = mans_amd.Workspace(0)
    got = mans_amd.lorenzo_reconstruct(codes, idx, val, shape, EB, ws)
    ws.check()
    assert torch.equal(got.view(torch.int32).reshape(-1), want.view(torch.int32).reshape(-1))
    ws.close()
