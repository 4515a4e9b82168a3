"""Performance cases of the codec: what its users have it do, through the
public entry points of the Python package.

listed() gives the fixed cases, draw(rng) one more of the same ranges,
prepare(case, seed) the inputs and handles a user's program holds before the
call, run(state) one pass, work(case) the bytes a pass cannot do without, and
exact(case, seed) a field's 64-bit values where a pass computes numbers (the
Lorenzo inverse; every other output is integers or bytes).

Kinds:
  frame    one buffer of 1/2/4-byte elements coded as a frame and / or decoded
  stream   raw bytes as one single-stream container, the drop-in API
  batch    a planned batch of uneven buffers (the batched launch)
  serve    a burst of mixed requests to the request server
  lorenzo  the 3-D Lorenzo front end, forward or inverse
Values come from the generators of mans_amd.workloads or are Laplace.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import mans_amd
from mans_amd import workloads

MIB = 1 << 20
EB = 1e-3      # error bound of the Lorenzo front end
RADIUS = 512   # its code radius
DTYPES = {1: torch.int8, 2: torch.int16, 4: torch.int32}
MODES = {"planes": mans_amd.MODE_PLANES, "adm": mans_amd.MODE_ADM, "auto": mans_amd.MODE_AUTO}


def _frame(name, elem_bytes, n, values, direction, lanes=64, prob_bits=10, mode="planes", b=4.0, wait=True):
    """wait: the calls use their defaults (the size comes back to the host,
    the decoder reads the header itself); otherwise the size stays on the
    device and the decoder is given the header, so nothing synchronises."""
    return {"name": name, "kind": "frame", "elem_bytes": elem_bytes, "n": n, "values": values,
            "direction": direction, "lanes": lanes, "prob_bits": prob_bits, "mode": mode, "b": b, "wait": wait}


def listed():
    return [
        # the smallest calls: a log record or a small message, where launches
        # and host work are all there is
        _frame("frame_u8_12k", 1, 12_289, "laplace", "both", prob_bits=11, b=9.0),
        # the small single-buffer configuration: 2,097,152 uint16 values
        _frame("frame_u16_4m", 2, 2_097_152, "laplace", "both"),
        # ordinary, ragged: a few image planes of 32-bit words, all of an
        # element's four planes coded (the Zipf configuration at a quarter)
        _frame("frame_u32_zipf_128m", 4, 33_554_431, "zipf", "both"),
        # the largest: 1 GiB of Lorenzo quantisation codes of a simulation
        # field, encoded on the device without waiting (the headline input)
        _frame("frame_codes_1g_encode", 2, 1 << 29, "codes", "encode", wait=False),
        # the same read back, a ragged size
        _frame("frame_codes_800m_decode", 2, 419_430_397, "codes", "decode", wait=False),
        # detector frames through the ADM byte mapping, both directions
        # (64 frames of 2048 x 2048)
        _frame("frame_detector_adm", 2, 64 * 2048 * 2048, "detector", "both", mode="auto"),
        # the drop-in 32-lane stream API on raw bytes, both directions
        {"name": "stream_bytes_256m", "kind": "stream", "n": 268_435_455, "lanes": 32, "prob_bits": 10},
        # batched form: uneven buffers of all widths in one launch, each way
        {"name": "batch_encode", "kind": "batch", "count": 1024, "lo": 4096, "hi": 4 * MIB, "lanes": 64,
         "prob_bits": 10, "direction": "encode"},
        {"name": "batch_decode", "kind": "batch", "count": 1024, "lo": 4096, "hi": 4 * MIB, "lanes": 64,
         "prob_bits": 10, "direction": "decode"},
        # served form: a burst of mixed compress / decompress requests
        {"name": "serve_burst", "kind": "serve", "count": 64, "lo": 64 << 10, "hi": 32 * MIB, "prob_bits": 10},
        # the error-bounded front end: field to codes and outliers, and back
        # (the inverse on a ragged field)
        {"name": "lorenzo_forward", "kind": "lorenzo", "nz": 512, "ny": 512, "nx": 1024, "direction": "forward"},
        {"name": "lorenzo_inverse", "kind": "lorenzo", "nz": 500, "ny": 499, "nx": 900, "direction": "inverse"},
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    kind = rng.choices(["frame", "stream", "batch", "serve", "lorenzo"], [8, 2, 3, 1, 2])[0]
    if kind == "frame":
        eb = rng.choice([1, 2, 2, 4])
        n = max(1, _log_uniform(rng, 4096, 512 * MIB) // eb)
        if rng.random() < 0.25:
            n = max(1, n & ~8191)  # whole blocks
        values = rng.choice(["laplace", "zipf"] if eb != 2 else ["laplace", "zipf", "codes", "detector"])
        mode = "auto" if eb == 2 and values in ("laplace", "detector") and rng.random() < 0.5 else "planes"
        c = _frame("", eb, n, values, rng.choice(["encode", "decode", "both"]), rng.choice([64, 64, 32]),
                   rng.choice([9, 10, 10, 11]), mode, round(math.exp(rng.uniform(0.0, math.log(64.0))), 3),
                   rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "stream":
        return {"kind": "stream", "n": _log_uniform(rng, 4096, 512 * MIB), "lanes": rng.choice([32, 32, 64]),
                "prob_bits": rng.choice([9, 10, 10, 11])}
    if kind == "batch":
        return {"kind": "batch", "count": _log_uniform(rng, 4, 1024), "lo": 4096,
                "hi": _log_uniform(rng, 64 << 10, 4 * MIB), "lanes": rng.choice([64, 64, 32]),
                "prob_bits": rng.choice([9, 10, 10, 11]), "direction": rng.choice(["encode", "decode"])}
    if kind == "serve":
        return {"kind": "serve", "count": _log_uniform(rng, 4, 64), "lo": 64 << 10,
                "hi": _log_uniform(rng, MIB, 32 * MIB), "prob_bits": 10}
    return {"kind": "lorenzo", "nz": _log_uniform(rng, 24, 512), "ny": _log_uniform(rng, 24, 512),
            "nx": _log_uniform(rng, 32, 1024), "direction": rng.choice(["forward", "inverse"])}


# ---- inputs ------------------------------------------------------------------
def _wrap(v, bits):
    """int64 values of `bits`-bit unsigned numbers as the signed type of that
    width (same bits)."""
    return torch.where(v >= (1 << (bits - 1)), v - (1 << bits), v).to(DTYPES[bits // 8])


def _laplace(n, eb, b, seed):
    """clip(half range + round(Laplace(0, b))) of n elements of eb bytes."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    bits = 8 * eb
    out = torch.empty(n, dtype=DTYPES[eb], device="cuda")
    for i in range(0, n, 1 << 24):
        m = min(1 << 24, n - i)
        u = torch.rand(m, generator=g, device="cuda", dtype=torch.float64) - 0.5
        lap = -b * torch.sign(u) * torch.log1p(-2.0 * u.abs())
        out[i:i + m] = _wrap(torch.clamp(torch.round(lap).to(torch.int64) + (1 << (bits - 1)), 0, (1 << bits) - 1),
                             bits)
    return out


def _dual_quant(field):
    """Codes and outliers of a field: q = rint(f / 2 EB) in float32, its 3-D
    Lorenzo residual r, code 32768 + r, or 0 with r an outlier."""
    q = torch.round(field * np.float32(1.0 / (2.0 * EB)).item()).to(torch.int32)
    for dim in range(3):
        low = torch.zeros_like(q)
        low.narrow(dim, 1, q.shape[dim] - 1).copy_(q.narrow(dim, 0, q.shape[dim] - 1))
        q -= low
    r = q.reshape(-1)
    inside = r.abs() < RADIUS
    idx = torch.nonzero(~inside).reshape(-1)
    val = r[idx].contiguous()
    # 32768 + r in 16 bits, as the signed type of the same bits
    codes = torch.where(inside, torch.where(r >= 0, r - 32768, r + 32768), torch.zeros_like(r)).to(torch.int16)
    return codes, idx.to(torch.int32), val


def _values(case, seed):
    n, eb = case["n"], case["elem_bytes"]
    if case["values"] == "laplace":
        return _laplace(n, eb, case["b"], seed)
    if case["values"] == "zipf":
        v = workloads.zipf_u32(n, seed=seed)
        return v if eb == 4 else _wrap(v.to(torch.int64) & ((1 << (8 * eb)) - 1), 8 * eb)
    if case["values"] == "detector":
        frames = -(-n // (2048 * 2048))
        return workloads.detector_u16(frames, 2048, seed)[:n].clone()
    ny = min(512, max(8, n // 8192))
    field = workloads.sinusoid_field((max(1, -(-n // (ny * 1024))), ny, 1024), seed)
    return _dual_quant(field)[0][:n].clone()


def _buffers(case, seed):
    """Uneven buffers: sizes log-uniform in [lo, hi] bytes, element width 1 / 2
    / 4 at 20 / 60 / 20 %, values 50 / 50 Laplace (b log-uniform in [1, 64]) or
    Zipf.  Sizes, widths and sources belong to the case, values to the seed."""
    rng = np.random.default_rng(1000 + case["count"])
    plan = []
    for _ in range(case["count"]):
        eb = int(rng.choice([1, 2, 4], p=[0.2, 0.6, 0.2]))
        nbytes = int(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]))))
        plan.append((max(1, nbytes // eb), eb, bool(rng.random() < 0.5), float(np.exp(rng.uniform(0.0, np.log(64.0))))))
    zipf = workloads.zipf_u32(max(1, sum(n for n, _, lap, _ in plan if not lap)), seed=seed)
    xs, at = [], 0
    for i, (n, eb, lap, b) in enumerate(plan):
        if lap:
            xs.append(_laplace(n, eb, b, 4096 * seed + i))
        else:
            v = zipf[at:at + n]
            at += n
            xs.append(v.clone() if eb == 4 else _wrap(v.to(torch.int64) & ((1 << (8 * eb)) - 1), 8 * eb))
    return xs


def _arena(sizes):
    """One zeroed buffer and a 256-byte aligned view of each size in it."""
    at, offs = 0, []
    for n in sizes:
        offs.append(at)
        at += -(-max(1, n) // 256) * 256
    whole = torch.zeros(at, dtype=torch.uint8, device="cuda")
    return whole, [whole[o:o + max(1, n)] for o, n in zip(offs, sizes)]


class _ArenaDecode(mans_amd.DecodeBatch):
    """A planned batch decode into the caller's own output buffers."""

    def __init__(self, frames, sizes, outs, xs, p, ws):
        self.keep = (frames, outs, ws)
        arr = (mans_amd.Buffer * len(frames))()
        for i, (f, size, o, x) in enumerate(zip(frames, sizes, outs, xs)):
            arr[i] = mans_amd.Buffer(f.data_ptr(), size, o.data_ptr(), o.numel(), x.numel(), x.element_size(), 0)
        self.handle = ctypes.c_void_p()
        rc = mans_amd.lib().mans_batch_decode_create(ctypes.byref(self.handle), ctypes.byref(p), arr, len(frames),
                                                     ws.handle)
        if rc:
            raise mans_amd.MansError(rc, "mans_batch_decode_create")

    def run(self, stream=None):
        s = stream if stream is not None else torch.cuda.current_stream()
        rc = mans_amd.lib().mans_batch_decode_run(self.handle, s.cuda_stream)
        if rc:
            raise mans_amd.MansError(rc, "mans_batch_decode_run")


def _field(case, seed):
    return workloads.sinusoid_field((case["nz"], case["ny"], case["nx"]), seed)


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case, "ws": mans_amd.Workspace(0)}
    ws = st["ws"]
    if kind == "frame":
        x = _values(case, seed)
        eb = case["elem_bytes"]
        p = mans_amd.params(case["prob_bits"], case["lanes"], eb, MODES[case["mode"]])
        ws.reserve(x.numel() * eb, p)
        st.update(x=x, p=p, n=x.numel(), dtype=x.dtype,
                  out=torch.zeros(mans_amd.frame_max_size(x.numel(), p), dtype=torch.uint8, device="cuda"),
                  d_size=torch.zeros(1, dtype=torch.int64, device="cuda"),
                  back=torch.zeros(max(8, x.numel()), dtype=x.dtype, device="cuda"))
        if case["direction"] == "decode":
            _, st["size"] = mans_amd.frame_encode(x, p, ws, out=st["out"])
            st["header"] = st["out"][:128].cpu().numpy().tobytes()
    elif kind == "stream":
        x = _laplace((case["n"] + 1) // 2, 2, 40.0, seed).view(torch.uint8)[:case["n"]]
        p = mans_amd.params(case["prob_bits"], case["lanes"])
        ws.reserve(x.numel(), p)
        st.update(x=x, p=p, n=x.numel(),
                  out=torch.zeros(mans_amd.max_compressed_size(x.numel(), p), dtype=torch.uint8, device="cuda"),
                  back=torch.zeros(x.numel(), dtype=torch.uint8, device="cuda"))
    elif kind == "batch":
        xs = _buffers(case, seed)
        p = mans_amd.params(case["prob_bits"], case["lanes"])
        caps = [mans_amd.frame_max_size(x.numel(), mans_amd.params(p.prob_bits, p.lanes, x.element_size())) for x in xs]
        whole, frames = _arena(caps)
        enc = mans_amd.EncodeBatch(xs, p, ws, outs=frames)
        st.update(batch=enc, whole=whole)
        if case["direction"] == "decode":
            sizes = enc.run().tolist()
            whole, outs = _arena([x.numel() * x.element_size() for x in xs])
            st.update(batch=_ArenaDecode(frames, sizes, outs, xs, p, ws), whole=whole)
    elif kind == "serve":
        xs = _buffers(case, seed)
        p = mans_amd.params(case["prob_bits"], 64)
        server = mans_amd.Server(p, 8 * 10**9)
        reqs, frames, caps = [], [], []
        for i, x in enumerate(xs):
            eb = x.element_size()
            if i % 2 == 0:
                reqs.append(server.compress_request(x))
                caps.append(mans_amd.frame_max_size(x.numel(), mans_amd.params(p.prob_bits, 64, eb)))
            else:
                f, size = mans_amd.frame_encode(x, p, ws)
                frames.append(f)
                reqs.append(server.decompress_request(f, size, x.numel(), eb))
                caps.append(x.numel() * eb)
        torch.cuda.synchronize()
        whole, outs = _arena(caps)
        st.update(xs=xs, frames=frames, server=server, reqs=reqs, whole=whole, outs=outs)
    elif case["direction"] == "forward":
        n = case["nz"] * case["ny"] * case["nx"]
        st["field"] = _field(case, seed)
        st["outliers"] = torch.zeros((2, max(1024, n // 64)), dtype=torch.int32, device="cuda")
    else:
        codes, idx, val = _dual_quant(_field(case, seed))
        st.update(codes=codes, idx=idx, val=val, shape=(case["nz"], case["ny"], case["nx"]))
    return st


def run(st):
    case, ws = st["case"], st["ws"]
    kind = st["kind"]
    if kind == "frame":
        outs = []
        size = st.get("size")
        if case["direction"] != "decode":
            if case["wait"] or case["direction"] == "both":
                outs += mans_amd.frame_encode(st["x"], st["p"], ws, out=st["out"])
                size = outs[1]
            else:
                outs += mans_amd.frame_encode(st["x"], st["p"], ws, out=st["out"], sync_size=False,
                                              d_size=st["d_size"])
        if case["direction"] != "encode":
            outs.append(mans_amd.frame_decode(st["out"], size, st["dtype"], st["n"], ws, out=st["back"],
                                              header=None if case["wait"] else st.get("header")))
        return outs
    if kind == "stream":
        out, size = mans_amd.encode(st["x"], st["p"], ws, out=st["out"])
        return [out, size, mans_amd.decode(out, st["n"], st["p"], ws, out=st["back"], c=size)]
    if kind == "batch":
        return [st["batch"].run(), st["whole"]][case["direction"] == "decode":]
    if kind == "serve":
        # results leave the server's memory for the program's own buffers as
        # they become ready
        server = st["server"]
        sizes = []
        for rid, out in zip(server.submit_many(st["reqs"]), st["outs"]):
            res = server.wait(rid)
            out[:res.out_bytes].copy_(server.fetch(res))
            server.release(rid)
            sizes.append(res.out_bytes)
        return [torch.tensor(sizes), st["whole"]]
    if case["direction"] == "forward":
        codes, idx, val = mans_amd.lorenzo_quantize(st["field"], EB, ws, radius=RADIUS)
        # into the program's outlier record
        st["outliers"][0, :idx.numel()] = idx
        st["outliers"][1, :idx.numel()] = val
        return [codes, idx.numel(), st["outliers"]]
    return mans_amd.lorenzo_reconstruct(st["codes"], st["idx"], st["val"], st["shape"], EB, ws)


# ---- work --------------------------------------------------------------------
def _bits_per_byte(values, eb, b):
    """About how many coded bits a byte of these values takes."""
    if values == "laplace":
        low = min(8.0, math.log2(2.0 * math.e * max(b, 0.5)))
        return (low if eb == 1 else (low + 1.0) / eb) + 0.25
    if values == "detector":
        return 3.0
    return 3.85 if values == "codes" else {1: 7.0, 2: 7.0, 4: 6.4}[eb]


def work(case):
    kind = case["kind"]
    if kind == "lorenzo":
        return {"bytes": 6 * case["nz"] * case["ny"] * case["nx"], "flops": 0}
    if kind == "frame":
        n = case["n"] * case["elem_bytes"]
        c = n * _bits_per_byte(case["values"], case["elem_bytes"], case["b"]) / 8.0
        passes = 2 if case["direction"] == "both" else 1
    elif kind == "stream":
        n, c, passes = case["n"], case["n"] * 0.6, 2
    else:
        n = case["count"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        c, passes = 0.66 * n, 1
    return {"bytes": int(passes * (n + c)), "flops": 0}


def exact(case, seed):
    if case["kind"] != "lorenzo" or case["direction"] != "inverse":
        return None
    codes, idx, val = _dual_quant(_field(case, seed))
    r = codes.to(torch.int64) + 32768
    r = torch.where(r >= 32768, r - 65536, r)
    r[codes == 0] = 0
    r[idx.to(torch.int64)] = val.to(torch.int64)
    r = r.reshape(case["nz"], case["ny"], case["nx"])
    for dim in range(3):
        r = torch.cumsum(r, dim)
    return r.to(torch.float64) * (2.0 * EB)
