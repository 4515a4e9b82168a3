"""A workspace frozen by a captured Lorenzo inverse serves what it would serve
with 4 bytes an element, whichever route the captured call took: fields of
another shape, a field that overlaps its codes, an ADM frame; no more than
that; and the graph keeps its own scratch."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402
from test_gpu_lorenzo_bands import EB, field  # noqa: E402

SHAPE = (64, 512, 256)  # 8 M elements by tiles: about 1.2 bytes an element
N = 64 * 512 * 256


def same(got, want):
    return torch.equal(got.view(torch.int32).reshape(-1), want.view(torch.int32).reshape(-1))


def frozen(codes, idx, val, smooth):
    """A workspace with a captured inverse of SHAPE, its graph and output.  (A
    byte-plane frame before it sizes what ADM frames need beside scratch.)"""
    ws = mans_amd.Workspace(0)
    mans_amd.frame_encode(smooth, mans_amd.params(10, 64, 2, mans_amd.MODE_PLANES), ws)
    out = mans_amd.lorenzo_reconstruct(codes, idx, val, SHAPE, EB, ws)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        mans_amd.lorenzo_reconstruct(codes, idx, val, SHAPE, EB, ws, out=out, stream=s)
    return ws, graph, out


def overlapping(codes, idx, val, shape, ws, stream=None):
    n = codes.numel()
    buf = torch.zeros(n, dtype=torch.float32, device="cuda")
    inside = buf.view(torch.int16)[n:]
    inside.copy_(codes)
    return mans_amd.lorenzo_reconstruct(inside, idx, val, shape, EB, ws, out=buf.view(shape), stream=stream)


@pytest.mark.parametrize("kind", ["flat", "overlap", "captured overlap", "adm frame"])
def test_frozen_workspace_keeps_its_promise(kind):
    codes, idx, val, want = field(SHAPE, 3)
    smooth = (20000 + torch.randint(-20, 20, (N,), device="cuda")).to(torch.int16)
    ws, graph, out = frozen(codes, idx, val, smooth)
    torch.cuda.synchronize()
    print(f"frozen scratch: {kind}", flush=True)
    if kind == "flat":
        flat = (N // 8192, 1, 8192)
        c, i, v, w = field((2, N // 8192 // 2, 8192), 4)
        assert same(mans_amd.lorenzo_reconstruct(c, i, v, (2, N // 8192 // 2, 8192), EB, ws), w)
        c, i, v, w = field(flat, 5)
        assert same(mans_amd.lorenzo_reconstruct(c, i, v, flat, EB, ws), w)
    elif kind == "overlap":
        assert same(overlapping(codes, idx, val, SHAPE, ws), want)
    elif kind == "captured overlap":
        buf = torch.zeros(N, dtype=torch.float32, device="cuda")
        inside = buf.view(torch.int16)[N:]
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        g2 = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g2, stream=s):
            mans_amd.lorenzo_reconstruct(inside, idx, val, SHAPE, EB, ws, out=buf.view(SHAPE), stream=s)
        for _ in range(3):
            inside.copy_(codes)
            torch.cuda.synchronize()
            g2.replay()
            torch.cuda.synchronize()
            assert same(buf, want)
    else:
        p = mans_amd.params(10, 64, 2, mans_amd.MODE_ADM)
        f, size = mans_amd.frame_encode(smooth, p, ws)
        other = mans_amd.Workspace(0)
        ref, ref_size = mans_amd.frame_encode(smooth, p, other)
        assert size == ref_size and torch.equal(f[:size], ref[:size])
        assert torch.equal(mans_amd.frame_decode(f, size, torch.int16, N, ws), smooth)
        other.close()
    # the promise ends at 4 bytes an element
    more = (65, 512, 256)
    c, i, v, w = field(more, 6)
    with pytest.raises(mans_amd.MansError) as e:
        overlapping(c, i, v, more, ws)
    assert e.value.status == 5  # MANS_ERR_CAPACITY
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want)
    ws.check()
    del graph
    ws.close()
