"""More work than one grid of resident workgroups holds, so that workgroups
take second and later items: encode slots used again and tickets placed late,
ADM areas used in turn with tickets mapped twice among them, and decode items
whose LUTs replace another buffer's."""
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402

DT = {1: torch.int8, 2: torch.int16, 4: torch.int32}
NP = {1: np.uint8, 2: np.uint16, 4: np.uint32}
THREADS = min(16, len(os.sched_getaffinity(0)))


def values(n, eb, seed):
    """Elements whose spread changes along the input (units of all sizes)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    out = torch.empty(n, dtype=DT[eb], device="cuda")
    for i in range(0, n, 1 << 25):
        m = min(1 << 25, n - i)
        k = torch.arange(i, i + m, device="cuda") // 50_000
        x = torch.randn(m, generator=g, device="cuda") * (0.2 + (k % 13).to(torch.float32) * 3.0)
        out[i:i + m] = x.to(torch.int32).to(DT[eb])
    return out


# elements: a ticket is 8 or 16 units of 8192 symbols (16 or 32 of 4096 at 32
# lanes), a grid 768 to 1280 workgroups: more than three tickets each
@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("eb,n", [(1, 300_000_011), (2, 150_000_003), (4, 80_000_005)])
def test_encode_workgroups_take_several_tickets(eb, n, lanes):
    p = mans_amd.params(10, lanes, eb, mans_amd.MODE_PLANES)
    x = values(n, eb, eb + lanes)
    ws = mans_amd.Workspace(0)
    out, size = mans_amd.frame_encode(x, p, ws)
    print(f"encode {n} elements of {eb} bytes at {lanes} lanes: {size} bytes", flush=True)
    fmt = oracle.FORMAT_NATIVE if lanes == 64 else oracle.FORMAT_REF
    ref = oracle.frame_encode(x.cpu().numpy().view(NP[eb]), oracle.MODE_PLANES, 10, fmt, threads=THREADS)
    assert size == ref.size
    assert torch.equal(out[:size], torch.from_numpy(ref).cuda())
    assert torch.equal(mans_amd.frame_decode(out, size, DT[eb], n, ws), x)
    ws.check()
    ws.close()


def test_adm_workgroups_take_several_tickets():
    # narrow stretches, lanes too long for a register, and stretches whose
    # bits exceed a wavefront's area (mapped again, when a later ticket has
    # been mapped already): 1832 tickets of 65,536 elements
    n = 120_000_123
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    x = torch.randn(n, generator=g, device="cuda") * 8.0
    k = torch.arange(n, device="cuda") // 30_000
    wide = k % 3 == 1
    x[wide] = torch.clamp(x[wide] * 40.0, -1500.0, 1500.0)
    x[torch.randint(0, n, (n // 7000,), generator=g, device="cuda")] += 3000.0
    x = (20000.0 + x).to(torch.int32).to(torch.int16)
    del k, wide
    gs = (n + 511) // 512
    ws = mans_amd.Workspace(0)
    ok, offs, cen, codes, bits = mans_amd.adm_map(x, ws)
    print(f"adm map {n} elements: {bits.numel()} bytes of bits", flush=True)
    rok, roffs, rcen, rcodes, rbits = oracle.adm_map(x.cpu().numpy().view(np.uint16))
    assert ok and rok
    for got, ref in ((offs[:gs + 1], roffs), (cen[:gs], rcen.view(np.int16)), (codes[:n], rcodes)):
        assert torch.equal(got.reshape(-1), torch.from_numpy(ref).cuda().to(got.dtype)), ref.size
    assert torch.equal(bits[:rbits.size], torch.from_numpy(rbits).cuda())
    back = mans_amd.adm_unmap(offs, cen, codes, bits, n, ws)
    assert torch.equal(back, x)
    ws.check()
    ws.close()


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("p", [9, 10, 11])
def test_decode_workgroups_take_several_items(p, lanes):
    # 9000 buffers of one to five tickets, neighbours of other widths and
    # spreads: every workgroup of the grid rebuilds its LUTs several times
    count, block = 9000, 128 * lanes
    rng = np.random.default_rng(p)
    xs, at = [], 0
    pool = {eb: values(1 << 24, eb, 40 + eb) for eb in DT}
    for i in range(count):
        eb = int(rng.choice([1, 2, 4]))
        n = int(rng.integers(1, 5 * block // (1 if eb == 1 else 2) + 2))
        at = (at + 50_000 + 16) % ((1 << 24) - 8 * block) // 16 * 16
        xs.append(pool[eb][at:at + n])
    ws = mans_amd.Workspace(0)
    par = mans_amd.params(p, lanes)
    enc = mans_amd.EncodeBatch(xs, par, ws)
    sizes = enc.run().tolist()
    print(f"decode {count} buffers at p {p}, {lanes} lanes", flush=True)
    dec = mans_amd.DecodeBatch(enc.outs, sizes, xs, par, ws)
    for _ in range(2):
        got = dec.run()
        ws.check()
        bad = torch.stack([(a != b).any() for a, b in zip(got, xs)])
        assert not bool(bad.any()), torch.nonzero(bad).reshape(-1).tolist()[:8]
        for t in got:
            t.zero_()
    dec.close()
    enc.close()
    ws.close()
