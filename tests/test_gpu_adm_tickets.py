"""ADM map and unmap at the edges of their tickets (a workgroup: 128 groups of
512 elements, a wavefront 32 of them, two at a time) and of the forms a lane's
bits take: a register word (all of a pair's lanes short), LDS atomics (one
lane long, or a partial group), a second mapping (more bytes than the
wavefront's area); unmap by words of 32 and 64 bits and by longer ones.  The
bit plane may start at any byte, and a short one is reported."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import mans_amd  # noqa: E402


def data(kind: str, n: int) -> np.ndarray:
    rng = np.random.default_rng(n + len(kind))
    x = 20000 + np.round(rng.normal(0, 8, n)).astype(np.int64)
    if kind == "flat":
        x[:] = 777
    elif kind == "edge":  # signals one step apart at each multiple of 126
        x = 20000 + rng.integers(-3, 4, n) * 126 + rng.integers(-1, 2, n)
    elif kind == "spikes":  # a long lane in a few pairs
        x[rng.integers(0, n, max(1, n // 5000))] += 3000
    elif kind == "wide":  # lanes of 5 to 32 bytes: more than the area holds
        x = 30000 + np.round(np.clip(rng.laplace(0, 250, n), -1500, 1500)).astype(np.int64)
    elif kind == "mixed":  # narrow and wide stretches
        w = (np.arange(n) // 4096) % 3 == 1
        x[w] = 30000 + np.round(np.clip(rng.laplace(0, 250, int(w.sum())), -1500, 1500)).astype(np.int64)
    elif kind == "ends":
        x = np.where(rng.random(n) < 0.5, rng.integers(0, 120, n), rng.integers(0, 300, n))
    return x.astype(np.uint16)


SIZES = [15, 16, 1023, 1024, 1025, 16384, 16385, 65535, 65536, 65537, 65536 + 16384 - 1, 3 * 65536 + 512 * 33 + 7]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("kind", ["narrow", "flat", "edge", "spikes", "wide", "mixed", "ends"])
def test_map_and_unmap_match_the_oracle(kind, shift):
    ws = mans_amd.Workspace(0)
    for n in SIZES:
        x = data(kind, n)
        print(f"adm {kind} n={n} shift={shift}", flush=True)
        g = (n + 511) // 512
        t = torch.from_numpy(np.concatenate([x, np.zeros(-n % 8, np.uint16)]).view(np.int16)).cuda()[:n]
        offs = torch.empty(g + 1, dtype=torch.int32, device="cuda")
        cen = torch.empty(g, dtype=torch.int16, device="cuda")
        codes = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
        bits = torch.full((g * 1024 + 32,), 0x5a, dtype=torch.uint8, device="cuda")
        blen, dom = ctypes.c_uint64(0), ctypes.c_int32(0)
        s = torch.cuda.current_stream().cuda_stream

        def call(cap):
            return mans_amd.lib().mans_adm_map(t.data_ptr(), n, offs.data_ptr(), cen.data_ptr(), codes.data_ptr(),
                                               bits.data_ptr() + shift, cap, ctypes.byref(blen), ctypes.byref(dom),
                                               ws.handle, s)

        rok, roffs, rcen, rcodes, rbits = oracle.adm_map(x)
        assert call(g * 1024) == 0 and bool(dom.value) == rok
        assert rok and blen.value == rbits.size
        got = bits.cpu().numpy()
        assert (offs.cpu().numpy() == roffs).all() and (cen.cpu().numpy().view(np.uint16) == rcen).all()
        assert (codes.cpu().numpy()[:n] == rcodes).all()
        assert (got[shift:shift + rbits.size] == rbits).all()
        assert (got[:shift] == 0x5a).all() and (got[shift + rbits.size:] == 0x5a).all()
        back = mans_amd.adm_unmap(offs, cen, codes, bits[shift:], n, ws).cpu().numpy().view(np.uint16)
        assert (back == x).all()
        # one byte too few: reported, nothing written past the end
        bits.fill_(0x5a)
        assert call(rbits.size - 1) == 5  # MANS_ERR_CAPACITY
        assert (bits.cpu().numpy()[shift + rbits.size - 1:] == 0x5a).all()
    ws.close()
