"""A result fetched on a busy stream and released at once: the copy is still
enqueued when the memory goes back, so no later request may be launched into
it before the copy has run."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402


def values(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return (torch.randn(n, generator=g, device="cuda") * 9).to(torch.int8)


@pytest.mark.parametrize("room", ["plenty", "one result"])
def test_release_with_the_copy_enqueued(room):
    p = mans_amd.params(10, 64)
    n = 64 << 20
    budget = 8_000_000_000
    if room == "one result":  # arena memory for one output at a time
        probe = mans_amd.Server(p, budget)
        own = budget - probe.stats()["arena_bytes"]
        probe.close()
        budget = own + 3 * n // 2 + (64 << 20)
    xs = [values(n, i) for i in range(4)]
    ws = mans_amd.Workspace(0)
    want = []
    for x in xs:
        f, size = mans_amd.frame_encode(x, mans_amd.params(10, 64, 1, mans_amd.MODE_PLANES), ws)
        want.append(f[:size].clone())
    srv = mans_amd.Server(p, budget)
    busy = torch.zeros(1 << 28, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    got = []
    for i, x in enumerate(xs):
        rid = srv.submit_compress(x)
        res = srv.wait(rid, 60_000)
        assert res is not None and res.status == 0
        for _ in range(100):  # some 50 ms of work before the copy
            busy.add_(1)
        got.append(srv.fetch(res))
        srv.release(rid)
        print(f"server release ({room}): request {i}", flush=True)
    torch.cuda.synchronize()
    for i, (g, w) in enumerate(zip(got, want)):
        assert torch.equal(g, w), i
    assert srv.stats()["arena_used"] == 0
    srv.close()
    ws.check()
    ws.close()


@pytest.mark.parametrize("stream", ["default", "own", "thread"])
def test_release_after_gives_the_memory_back(stream):
    # (2: hipStreamPerThread, which only the releasing thread can record on)
    own = torch.cuda.Stream()
    handle = {"default": 0, "own": own.cuda_stream, "thread": 2}[stream]
    srv = mans_amd.Server(mans_amd.params(10, 64), 4 << 30)
    x = values(1 << 20, 3)
    torch.cuda.synchronize()
    rid = srv.submit_compress(x)
    assert srv.wait(rid, 60_000).status == 0
    assert srv.stats()["arena_used"] > 0
    assert mans_amd.lib().mans_server_release_after(srv.handle, rid, handle) == 0
    assert mans_amd.lib().mans_server_release_after(srv.handle, rid, handle) == 1  # (released: unknown)
    torch.cuda.synchronize()
    assert srv.stats()["arena_used"] == 0
    srv.close()
