"""Batched decode of a frame with a malformed table in any one plane: the
buffer is flagged and nothing of it is written, its neighbours decode."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

DT = {1: torch.uint8, 2: torch.int16, 4: torch.int32}


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("eb,plane", [(1, 0), (2, 0), (2, 1), (4, 0), (4, 1), (4, 2), (4, 3)])
def test_a_bad_table_rejects_the_whole_buffer(eb, plane, lanes):
    n = 40 * 128 * lanes + 77
    g = torch.Generator(device="cuda")
    g.manual_seed(eb * 10 + plane)
    xs = [torch.randint(0, 200, (n,), generator=g, device="cuda").to(DT[eb]) for _ in range(3)]
    ws = mans_amd.Workspace(0)
    p = mans_amd.params(10, lanes)
    enc = mans_amd.EncodeBatch(xs, p, ws)
    sizes = enc.run().tolist()
    frames = [f[:s].clone() for f, s in zip(enc.outs, sizes)]
    # the plane's section begins at the offset in frame word 64 + 8 plane; its
    # table of uint16 frequencies after 32 bytes
    at = int(frames[1][64 + 8 * plane:72 + 8 * plane].view(torch.int64)[0]) + 32
    frames[1][at:at + 2].view(torch.int16).add_(1)
    print(f"batch decode: bad table of plane {plane}, {eb} bytes, {lanes} lanes", flush=True)
    dec = mans_amd.DecodeBatch(frames, sizes, xs, p, ws)
    for o in dec.outs:
        o.fill_(99)
    for _ in range(2):
        got = dec.run()
        torch.cuda.synchronize()
        flags = dec.flags()
        assert flags[0] == 0 and flags[1] != 0 and flags[2] == 0
        assert torch.equal(got[0], xs[0]) and torch.equal(got[2], xs[2])
        assert bool((got[1] == 99).all())
    with pytest.raises(mans_amd.MansError):
        ws.check()
    dec.close()
    enc.close()
    ws.close()
