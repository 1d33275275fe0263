"""The work that users of the X-engine have it do, as cases that can be timed and compared.

A correlator's pass is: start an integration, correlate the blocks that arrive, dump the
visibilities.  Three more kinds of pass go round it: the host-buffer pipeline of xgpu.h callers,
the serving loop of many subarrays, and the channelizer's FFTs.  Sizes are those of the library's
build variants, of bench.py and of workloads.serving_mix, or generic ones; array sizes in use run
from a dozen stations (a lab or test array) over tens and hundreds to two thousand.
"""
import numpy as np
import torch

import xgpu_amd as X
from xgpu_amd import workloads

COMPUTE = {"int8": X.XGPU_INT8, "fp16": X.XGPU_FLOAT16, "fp32": X.XGPU_FLOAT32}
ORDER = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER,
         "tri": X.TRIANGULAR_ORDER}


def _corr(name, nstation, nfrequency, ntime, **more):
    """calls: blocks of ntime samples in one integration; layout: plain, swizzled (the DP4A input's
    corner turn) or block32; data: uniform bytes, or sky (Gaussian noise plus a tone); wide: the
    64-bit dump; full: the dump is expanded to the full matrix too."""
    c = {"kind": "correlate", "name": name, "nstation": nstation, "nfrequency": nfrequency,
         "ntime": ntime, "compute": "int8", "order": "regtile", "layout": "plain",
         "data": "sky", "calls": 1, "wide": False, "full": False}
    c.update(more)
    return c


def listed():
    return [
        # a lab or test array: one small block, where launches and latency count
        _corr("int8_16st", 16, 2, 64),
        # the library's default sizing, one block of a 256-station array
        _corr("int8_256st", 256, 10, 1024),
        # bench.py's workload: one integration of a 512-station array on full-range bytes
        _corr("int8_512st", 512, 64, 8192, data="uniform"),
        # the largest array: a long input and a dump of a gigabyte
        _corr("int8_2048st", 2048, 16, 4096),
        # a ragged array (not a whole number of 4-station groups), odd channel count and block
        # length, split-plane order, and an imager behind it that reads full matrices
        _corr("int8_202st_full", 202, 37, 1001, order="realimag", calls=2, full=True),
        # a long integration of short blocks, past the 32-bit bound, dumped in 64 bits
        _corr("int8_96st_long", 96, 24, 2048, calls=40, wide=True),
        # input in the DP4A build's swizzled layout
        _corr("int8_352st_swizzled", 352, 29, 2048, layout="swizzled", calls=2),
        # half-precision voltages
        _corr("fp16_256st", 256, 128, 2048, compute="fp16"),
        # the float build of the library (int8 in, float visibilities) at its default sizing
        _corr("fp32_256st", 256, 10, 1024, compute="fp32"),
        # the host-buffer pipeline of an xgpu.h program at the library's default sizing
        {"kind": "host", "name": "host_256st", "nstation": 256, "nfrequency": 10, "ntime": 1024,
         "pipes": 8},
        # eight subarrays served at once from blocks in HBM, dumps left in HBM
        {"kind": "serve", "name": "serve_8", "mix": 5, "streams": 8, "shorten": 4},
        # a channelizer's transforms: the analysis of one block, the synthesis of another
        {"kind": "fft", "name": "fft_1024", "n": 1024, "batch": 8192, "layout": "natural"},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _mix(case):
    """(nstation, nfrequency, ntime, blocks per dump) of each stream."""
    mix = workloads.serving_mix(case["mix"], spill_stream=False)[:case["streams"]]
    return [(ns, nf, nt, max(1, k // case["shorten"])) for ns, nf, nt, k in mix]


def draw(rng):
    while True:
        kind = rng.choice(["int8", "int8", "int8", "int8", "fp16", "fp32", "swizzled", "block32",
                           "host", "serve", "fft", "fft"])
        if kind == "fft":
            n = 1 << rng.randint(3, 13)
            layout = rng.choice(["natural", "natural", "prototype"])
            if layout == "prototype":
                n = n if n not in (32, 128) else 256
                group = {8: 64, 16: 64, 64: 8}.get(n, 1)
            else:
                group = 1
            batch = max(1, _log(rng, 1 << 12, 1 << 23) // n // group) * group
            return {"kind": "fft", "n": n, "batch": batch, "layout": layout}
        if kind == "serve":
            c = {"kind": "serve", "mix": rng.randint(0, 999), "streams": rng.randint(2, 8),
                 "shorten": rng.choice([4, 8, 16])}
        else:
            step = {"swizzled": 4, "block32": 16}.get(kind, 2)
            ns = max(16, _log(rng, 16, 2048) // step * step)
            nf, nt = _log(rng, 1, 128), _log(rng, 48, 8192)
            if kind == "host":
                pipes = rng.choice([1, 2, 4, 8])
                c = {"kind": "host", "nstation": ns, "nfrequency": nf,
                     "ntime": max(1, nt // pipes) * pipes, "pipes": pipes}
                if nf * ns * c["ntime"] * 4 > 1 << 26 or nf * ns * ns > 1 << 22:
                    continue
            else:
                order = rng.choice(["regtile", "regtile", "realimag", "tri"])
                c = _corr("", ns, nf, nt, order="realimag" if ns % 4 and order == "regtile" else order,
                          compute=kind if kind in ("fp16", "fp32") else "int8",
                          data=rng.choice(["sky", "sky", "uniform"]) if kind != "fp16" else "sky",
                          layout=kind if kind in ("swizzled", "block32") else "plain",
                          calls=rng.choice([1, 1, 2, 3, 8, 20]), wide=rng.random() < 0.3,
                          full=rng.random() < 0.2)
                del c["name"]
                if kind == "swizzled":
                    c["ntime"] = max(4, nt // 4 * 4)
        # no more work than the largest listed case's: 1.1e12 / 8 flops a byte apart
        w, most = work(c), 2.2e12
        if w["flops"] > (most if c.get("compute") != "fp32" else most / 16) or w["bytes"] > 1.4e9:
            continue
        return c


# ---- inputs ------------------------------------------------------------------
def _blocks(compute, data, calls, nt, nf, ns, seed):
    """[calls, nt, nf, ns, 2, 2] on the GPU: the voltages in time order."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dtype = torch.float16 if compute == "fp16" else torch.int8
    x = torch.empty((calls * nt, nf, ns, 2, 2), dtype=dtype, device="cuda")
    phase = 6.2831853 * torch.rand((nf, ns, 1), generator=g, device="cuda")
    step = max(1, (1 << 26) // (nf * ns * 4))
    for t0 in range(0, calls * nt, step):
        part = x[t0:t0 + step]
        if data == "uniform":
            part.copy_(torch.randint(-128, 128, part.shape, generator=g, device="cuda",
                                     dtype=torch.int8))
            continue
        v = torch.randn(part.shape, generator=g, device="cuda")
        v *= 16.0 if compute == "fp16" else 20.0
        t = torch.arange(t0, t0 + part.shape[0], device="cuda", dtype=torch.float32)
        tone = 0.0371 * t[:, None, None, None] + phase
        amp = 4.0 if compute == "fp16" else 8.0
        v[..., 0] += amp * torch.cos(tone)
        v[..., 1] += amp * torch.sin(tone)
        part.copy_(v if compute == "fp16" else v.round_().clamp_(-127, 127))
    return x.view(calls, nt, nf, ns, 2, 2)


def _laid_out(x, layout):
    calls, nt, nf, ns = x.shape[:4]
    if layout == "swizzled":  # [t/4][f][s][p][c][t%4]
        x = x.view(calls, nt // 4, 4, nf, ns, 2, 2).permute(0, 1, 3, 4, 5, 6, 2)
    elif layout == "block32":  # 32 real parts, then their 32 imaginary parts
        x = x.view(calls, nt, nf, ns // 16, 32, 2).transpose(-1, -2)
    return x.contiguous()


def _ints(compute):
    return compute == "int8"


class _View:
    """A server stream's device ring as a tensor; keeps the server that owns it."""

    def __init__(self, ring, count, server):
        self.keep = (ring, server)
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<i8", "version": 2,
                                         "data": (ring.ptr, False), "strides": None}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fft":
        n = case["n"] * case["batch"]
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        x = torch.randn((2, n), generator=g, device="cuda", dtype=torch.complex64)
        return {"case": case, "x": x, "work": torch.empty_like(x),
                "layout": X.FFT_NATURAL if case["layout"] == "natural" else X.FFT_PROTOTYPE}
    if kind == "serve":
        server = X.Server()
        streams = []
        for s, (ns, nf, nt, k) in enumerate(_mix(case)):
            blocks = _blocks("int8", "uniform", k, nt, nf, ns, seed * 16 + s)
            sid, ring = server.open_stream(ns, nf, k, dump_slots=1, dump_device=True)
            out = torch.as_tensor(_View(ring, nf * ns * (ns + 1) * 4, server), device="cuda")
            streams.append((sid, blocks, nt, out))
        torch.cuda.synchronize()
        return {"case": case, "server": server, "streams": streams}
    ns, nf, nt = case["nstation"], case["nfrequency"], case["ntime"]
    if kind == "host":
        x = _blocks("int8", "sky", 1, nt, nf, ns, seed)
        array_h = torch.empty(x.shape, dtype=torch.int8, pin_memory=True)
        array_h.copy_(x)
        eng = X.Engine(ns, nf, ntime=nt, ntimepipe=nt // case["pipes"], order=ORDER["tri"])
        matrix_h = torch.zeros(2 * eng.mat_len, dtype=torch.int32, pin_memory=True)
        torch.cuda.synchronize()
        return {"case": case, "eng": eng, "array_h": array_h, "matrix_h": matrix_h}
    x = _laid_out(_blocks(case["compute"], case["data"], case["calls"], nt, nf, ns, seed),
                  case["layout"])
    eng = X.Engine(ns, nf, compute=COMPUTE[case["compute"]], order=ORDER[case["order"]],
                   complex_block_size=32 if case["layout"] == "block32" else 1,
                   time_swizzle=4 if case["layout"] == "swizzled" else 0)
    if _ints(case["compute"]):
        dtype = torch.int64 if case["wide"] else torch.int32
    else:
        dtype = torch.float64 if case["wide"] else torch.float32
    state = {"case": case, "eng": eng, "x": x,
             "out": torch.empty(2 * eng.tri_len, dtype=dtype, device="cuda")}
    if case["full"]:
        state["matrix"] = torch.empty(nf * ns * ns * 8, dtype=dtype, device="cuda")
        state["elem"] = {torch.int32: X.ELEM_INT32, torch.int64: X.ELEM_INT64,
                         torch.float32: X.ELEM_FLOAT32, torch.float64: X.ELEM_FLOAT64}[dtype]
    torch.cuda.synchronize()
    return state


# ---- one pass -----------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fft":  # the work buffers are filled anew, as the stage before the FFT does
        stream = torch.cuda.current_stream().cuda_stream
        work = state["work"].copy_(state["x"])
        X.fft(work[0].data_ptr(), case["n"], case["batch"], False, state["layout"], stream)
        X.fft(work[1].data_ptr(), case["n"], case["batch"], True, state["layout"], stream)
        return {"spectrum": work[0], "signal": work[1]}
    if kind == "serve":
        server = state["server"]
        for b in range(max(blocks.shape[0] for _, blocks, _, _ in state["streams"])):
            for sid, blocks, nt, _ in state["streams"]:
                if b < blocks.shape[0]:
                    server.submit_device(sid, blocks[b].data_ptr(), nt)
        server.drain()
        return [out for _, _, _, out in state["streams"]]
    eng, lib = state["eng"], X.core()
    eng.clear()
    if kind == "host":
        X.check(lib.xgpuAmdCorrelateHost(eng.handle, state["array_h"].data_ptr(), X.SYNCOP_DUMP,
                                         state["matrix_h"].data_ptr()))
        return state["matrix_h"]
    for block in state["x"]:
        eng.correlate(block.data_ptr(), case["ntime"])
    flags = X.XGPU_DUMP_DEVICE | X.XGPU_DUMP_TRIANGULAR
    X.check(lib.xgpuAmdDump(eng.handle, state["out"].data_ptr(),
                            flags | (X.XGPU_DUMP_WIDE if case["wide"] else 0)))
    if not case["full"]:
        return state["out"]
    X.extract_matrix(state["matrix"].data_ptr(), state["out"].data_ptr(), case["nstation"],
                     case["nfrequency"], state["elem"])
    return {"packed": state["out"], "matrix": state["matrix"]}


# ---- what a pass cannot do without ----------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "fft":  # the usual 5 n log2(n) a transform
        n = case["n"] * case["batch"]
        return {"bytes": 2 * 2 * 8 * n, "flops": 2 * 5 * n * int(np.log2(case["n"]))}
    if kind == "serve":
        jobs = [(ns, nf, nt * k, 2, 8) for ns, nf, nt, k in _mix(case)]
    elif kind == "host":
        jobs = [(case["nstation"], case["nfrequency"], case["ntime"], 2, 4)]
    else:
        jobs = [(case["nstation"], case["nfrequency"], case["ntime"] * case["calls"],
                 4 if case["compute"] == "fp16" else 2, 8 if case["wide"] else 4)]
    nbytes = flops = 0
    for ns, nf, nt, cplx, elem in jobs:
        pairs = ns * (ns + 1) // 2
        nbytes += nf * nt * ns * 2 * cplx + nf * pairs * 8 * elem
        flops += 8 * X.cmac_per_integration(ns, nf, nt)
        if case.get("full"):
            nbytes += nf * ns * ns * 8 * elem
    return {"bytes": nbytes, "flops": flops}


# ---- the same in 64 bits --------------------------------------------------------
def _matrix64(x, wide_int):
    """Full visibility matrices [nf, ns, ns, 2, 2, 2] of voltages [nt, nf, ns, 2, 2]."""
    nt, nf, ns = x.shape[:3]
    for f in range(nf):
        re = im = 0.0
        step = max(1, (1 << 26) // (ns * 2))
        for t0 in range(0, nt, step):
            v = x[t0:t0 + step, f].reshape(-1, 2 * ns, 2).double()
            a, b = v[..., 0].t().contiguous(), v[..., 1].t().contiguous()
            at, bt = a.t().contiguous(), b.t().contiguous()
            re = re + a @ at + b @ bt
            im = im + b @ at - a @ bt
        v = torch.stack([re, im], -1).view(ns, 2, ns, 2, 2).permute(0, 2, 1, 3, 4)
        yield v.to(torch.int64) if wide_int else v


def _packed64(x, ints, full=False):
    nt, nf, ns = x.shape[:3]
    i, j = torch.tril_indices(ns, ns, device="cuda")
    kind = torch.int64 if ints else torch.float64
    packed = torch.empty((nf, i.numel(), 2, 2, 2), dtype=kind, device="cuda")
    matrix = torch.empty((nf, ns, ns, 2, 2, 2), dtype=kind, device="cuda") if full else None
    for f, v in enumerate(_matrix64(x, ints)):
        packed[f] = v[i, j]
        if full:
            matrix[f] = v
    return {"packed": packed.view(-1), "matrix": matrix.view(-1)} if full else packed.view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return [_packed64(_blocks("int8", "uniform", k, nt, nf, ns, seed * 16 + s).flatten(0, 1), True)
                for s, (ns, nf, nt, k) in enumerate(_mix(case))]
    if kind == "fft":
        return _fft64(case, prepare(case, seed)["x"].to(torch.complex128))
    ns, nf, nt = case["nstation"], case["nfrequency"], case["ntime"]
    if kind == "host":
        return _packed64(_blocks("int8", "sky", 1, nt, nf, ns, seed)[0], True).cpu()
    x = _blocks(case["compute"], case["data"], case["calls"], nt, nf, ns, seed).flatten(0, 1)
    return _packed64(x, _ints(case["compute"]), case["full"])


def _fft64(case, x):
    """Both transforms, through the layout of the work buffer (include/xgpu_fft.h)."""
    n, batch = case["n"], case["batch"]
    proto = case["layout"] == "prototype"

    def gather(v, spectrum):  # work buffer -> [batch, n]
        if proto and n in (8, 16):
            return v.view(-1, n, 64).transpose(1, 2).reshape(batch, n)
        if proto and n == 64:
            return v.view(-1, 8, 8, 8).transpose(1, 2).reshape(batch, n)
        if proto and n >= 2048 and spectrum:
            return v.view(batch, n // 512, 512).transpose(1, 2).reshape(batch, n)
        return v.view(batch, n)

    def scatter(v, spectrum):  # [batch, n] -> work buffer
        if proto and n in (8, 16):
            return v.view(-1, 64, n).transpose(1, 2).reshape(-1)
        if proto and n == 64:
            return v.view(-1, 8, 8, 8).transpose(1, 2).reshape(-1)
        if proto and n >= 2048 and spectrum:
            return v.view(batch, 512, n // 512).transpose(1, 2).reshape(-1)
        return v.reshape(-1)

    return {"spectrum": scatter(torch.fft.fft(gather(x[0], False)), True),
            "signal": scatter(torch.fft.ifft(gather(x[1], True), norm="forward"), False)}
