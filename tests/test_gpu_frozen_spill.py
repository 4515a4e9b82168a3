"""A workspace frozen by a captured encode serves byte-plane frames and streams
of every element width of the size it was sized for, with the bytes a
workspace of their own gives; and the graph replays as before."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

DT = {1: torch.int8, 2: torch.int16, 4: torch.int32}


def values(nbytes, eb, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return (torch.randn(nbytes // eb, generator=g, device="cuda") * 20).to(DT[eb])


def frozen(nbytes, eb, lanes, p, reserve):
    ws = mans_amd.Workspace(0)
    q = mans_amd.params(p, lanes, eb, mans_amd.MODE_PLANES)
    x = values(nbytes, eb, eb)
    if reserve:
        ws.reserve(nbytes, q)
    ref, size = mans_amd.frame_encode(x, q, ws)
    ref = ref[:size].clone()
    out = torch.empty(mans_amd.frame_max_size(x.numel(), q), dtype=torch.uint8, device="cuda")
    d_size = torch.zeros(1, dtype=torch.int64, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        mans_amd.frame_encode(x, q, ws, out=out, stream=s, sync_size=False, d_size=d_size)
    torch.cuda.synchronize()
    return ws, graph, (x, out, d_size, ref)  # (the graph reads x)


# bytes: a few blocks (one workgroup or two), and more than the chip holds
@pytest.mark.parametrize("reserve,nbytes", [(False, 8 * 8192), (False, 24 * 8192), (True, 256 << 20)])
@pytest.mark.parametrize("eb", [1, 2, 4])
@pytest.mark.parametrize("p,lanes", [(9, 64), (11, 64), (10, 32)])
def test_frozen_workspace_serves_every_width(eb, p, lanes, reserve, nbytes):
    print(f"frozen spill: width {eb} p {p} lanes {lanes} bytes {nbytes}", flush=True)
    ws, graph, (_x, out, d_size, ref) = frozen(nbytes, eb, lanes, p, reserve)
    for eb2 in (1, 2, 4):
        q = mans_amd.params(p, lanes, eb2, mans_amd.MODE_PLANES)
        x = values(nbytes, eb2, 10 + eb2)
        other = mans_amd.Workspace(0)
        want, size = mans_amd.frame_encode(x, q, other)
        if reserve:
            ws.reserve(nbytes, q)
        got, got_size = mans_amd.frame_encode(x, q, ws)
        assert got_size == size and torch.equal(got[:size], want[:size]), eb2
        assert torch.equal(mans_amd.frame_decode(got, size, DT[eb2], x.numel(), ws), x)
        other.close()
    for _ in range(3):
        out.zero_()
        d_size.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        n = int(d_size.item())
        assert n == ref.numel() and torch.equal(out[:n], ref)
    ws.check()
    del graph
    ws.close()
