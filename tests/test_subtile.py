"""Sub-tile real-Gram kernel (xg_xengine_rgk): 64 x 64-input tiles, samples
split over the workgroup's waves and, for small blocks, over slices.

CPU: every unit is scheduled exactly once; a model of the kernel's DMAs
(resource, lane offsets, LDS window), operand reads and stores stays inside
its buffers and stores every visibility once.  GPU: int8 bit-exact against the
integer oracle at tile edges, sample tails, slices and in batches with square-tile
jobs; fp16 arrays of the same sizes (square tiles) within the accumulation bound of
the FP64 oracle.
"""
import ctypes as C

import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush
from test_schedule import XG_NXCD, XgLaunch

ORDERS = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER,
          "tri": X.TRIANGULAR_ORDER}
FMT = {"i8": dict(row=128, chunks=8, bpi=2, kk=32, chunk=lambda slot, r: slot ^ (r & 6)),
       "f16": dict(row=256, chunks=16, bpi=4, kk=16, chunk=lambda slot, r: slot ^ ((r & 3) << 2))}
OOR = 0x7fffff00


def split_len(nt, s):
    return ((nt + s - 1) // s + 127) & ~127


@pytest.mark.parametrize("jobs", [[(64, 8, 1)], [(16, 2, 16)], [(84, 1, 4)], [(96, 116, 1)],
                                  [(4, 1, 1)], [(660, 3, 2)], [(96, 5, 1), (200, 3, 1), (16, 9, 1)]])
def test_every_unit_once(jobs):
    L = XgLaunch()
    for i, (ns, nf, split) in enumerate(jobs):
        J = L.jobs[i]
        J.nstation, J.nfreq, J.ntime = ns, nf, 64
        J.nblk = (2 * ns + 63) // 64
        J.pair_tiles = 2 | (split << 8)
        J.tiles_per_chan = J.nblk * (J.nblk + 1) // 2 * split
    L.njobs = len(jobs)
    lib = X.core()
    lib.xg_plan_launch.argtypes = [C.POINTER(XgLaunch), C.c_int, C.c_int]
    lib.xg_plan_launch(C.byref(L), 256, 1)
    lib.xgh_schedule.argtypes = [C.POINTER(XgLaunch), C.c_int, C.c_int] + [C.POINTER(C.c_int)] * 4
    seen, shares = [], []
    for x in range(XG_NXCD):
        k, v = 0, [C.c_int() for _ in range(4)]
        while lib.xgh_schedule(C.byref(L), x, k, *[C.byref(a) for a in v]):
            seen.append(tuple(a.value for a in v))
            k += 1
        shares.append(k)
    want = {(i + 16 * s, f, rb, cb) for i, (ns, nf, split) in enumerate(jobs) for s in range(split)
            for f in range(nf) for rb in range((2 * ns + 63) // 64) for cb in range(rb + 1)}
    assert len(seen) == len(want) and set(seen) == want
    assert max(shares) - min(shares) <= len(jobs)   # the XCDs are even
    assert L.wg_per_xcd == max(shares)              # one unit per workgroup


def model_unit(fmt, ns, nf, nt, f, rb, cb, split, nsplit):
    """Every DMA of the unit's 4 waves: in-range lanes read inside the block."""
    F = FMT[fmt]
    ts, ninput, K = nf * ns * 2 * F["bpi"], 2 * ns, F["kk"]
    t0 = split * split_len(nt, nsplit) if nsplit > 1 else 0
    n_t = min(nt - t0, split_len(nt, nsplit)) if nsplit > 1 else nt
    assert n_t > 0
    total, spd = nt * ts, 1024 // F["row"]
    lanes = np.arange(64)
    srow, slot = lanes // F["chunks"], lanes % F["chunks"]
    chunk = np.array([F["chunk"](int(a), int(b)) for a, b in zip(slot, srow)])
    for r in range(spd):  # the swizzle permutes a row's chunks
        assert sorted(chunk[srow == r]) == list(range(F["chunks"]))
    for wave in range(4):
        n = max(((n_t + K - 1) // K - wave + 3) >> 2, 1)
        n += n & 1
        for it in range(n + 4):
            k0 = (4 * it + wave) * K
            rows = max(min(n_t - k0, K), 0)
            for blk in {rb, cb}:
                nbytes = min(F["row"], (ninput - 64 * blk) * F["bpi"])
                base = t0 * ts + f * ninput * F["bpi"] + blk * F["row"] + k0 * ts
                nrec = rows * ts - ts + nbytes if rows > 0 else 0
                got = np.zeros((K, F["chunks"]), dtype=int)
                for j in range(4):
                    voff = np.where(16 * chunk < nbytes, (j * spd + srow) * ts + 16 * chunk, OOR)
                    ok = voff < nrec
                    a = base + voff[ok]
                    # whole 16 bytes in the block, or cut at the resource's end
                    end = np.minimum(a + 16, base + nrec)
                    assert (a >= 0).all() and (end <= total).all()
                    np.add.at(got, ((j * spd + srow)[ok], chunk[ok]), 1)
                assert (got[:rows, :(nbytes + 15) // 16] == 1).all()
                assert got.sum() == rows * ((nbytes + 15) // 16)


@pytest.mark.parametrize("fmt", ["i8", "f16"])
@pytest.mark.parametrize("ns,nf,nt,nsplit", [(4, 1, 1, 1), (16, 2, 64, 1), (36, 3, 33, 1),
                                             (64, 2, 129, 1), (68, 1, 700, 3), (96, 2, 257, 2),
                                             (132, 1, 515, 1)])
def test_loads_in_bounds(fmt, ns, nf, nt, nsplit):
    nb = (2 * ns + 63) // 64
    for f in {0, nf - 1}:
        for rb in range(nb):
            for cb in range(rb + 1):
                for s in range(nsplit):
                    model_unit(fmt, ns, nf, nt, f, rb, cb, s, nsplit)


@pytest.mark.parametrize("ns", [2, 4, 34, 36, 64, 100, 130])
@pytest.mark.parametrize("order", ["regtile", "realimag", "tri"])
def test_every_visibility_stored_once(ns, order):
    """rg_store_cells over 64-input tiles: cell (i, j) of wave w, lane and step."""
    if order == "regtile" and ns % 4:
        pytest.skip("register-tile order needs whole 4-station groups")
    half, nb2 = ns // 2, ns * (ns + 1) // 2
    per = half * (half + 1) // 2 if order == "regtile" else nb2
    plane = 16 * per if order == "regtile" else 4 * nb2
    hits = np.zeros(2 * plane, dtype=int)
    lane = np.arange(64)
    hi, mj, bq = lane >> 5, (lane & 31) >> 2, lane & 3
    nb = (2 * ns + 63) // 64
    for rb in range(nb):
        for cb in range(rb + 1):
            full = rb != cb and rb * 32 + 32 <= ns
            for w in range(4):
                j = cb * 32 + mj + 8 * (bq ^ w)
                for q in range(4):
                    I = rb * 32 + 8 * w + 2 * q
                    i = I + hi
                    keep = np.ones(64, bool)
                    if not full:
                        keep = (i < ns) & (j < ns) & ((i >= j) | ((order == "regtile") & (i >> 1 == j >> 1)))
                    assert (i[keep] < ns).all() and (j[keep] < ns).all()
                    if order == "regtile":
                        cell = (2 * (j & 1) + hi) * per + (j >> 1) + (I >> 1) * ((I >> 1) + 1) // 2
                    else:
                        cell = j + I * (I + 1) // 2 + hi * (I + 1)
                    for c in cell[keep]:
                        if order == "tri":
                            hits[8 * c:8 * c + 8] += 1
                        else:
                            hits[4 * c:4 * c + 4] += 1
                            hits[plane + 4 * c:plane + 4 * c + 4] += 1
    assert (hits == 1).all()


# a single partial tile, whole tiles, tile edges +- one group, sample tails,
# fewer ksteps than waves, more than the ring holds, blocks cut into slices
GPU_CASES = [(4, 1, 1), (16, 2, 64), (32, 3, 33), (60, 2, 129), (68, 1, 513), (96, 2, 257),
             (64, 2, 3000), (36, 1, 5003)]


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["regtile", "realimag", "tri"])
@pytest.mark.parametrize("ns,nf,nt", GPU_CASES)
def test_int8_exact(ns, nf, nt, order):
    flush(f"[sub-tiles] int8 ns={ns} nf={nf} nt={nt} {order}")
    x = oracle.fill_uniform(2 * nt * nf * ns * 4, 71, -128, 127)
    half = nt * nf * ns * 4
    bufs = [X.DeviceBuffer.from_array(x[:half]), X.DeviceBuffer.from_array(x[half:])]
    eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=ORDERS[order])
    for calls in (1, 2):  # stored, then accumulated
        eng.correlate(bufs[calls - 1], nt)
        got = eng.dump(wide=True, triangular=True)
        ref = oracle.xengine_i64(x[:calls * half], ns, nf, calls * nt)
        assert np.array_equal(got, ref), calls
    raw = eng.dump()
    eng.set_tuning(kernel=1)  # the general path, in the engine's own order
    eng.clear()
    for b in bufs:
        eng.correlate(b, nt)
    assert np.array_equal(raw, eng.dump())


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["regtile", "tri"])
@pytest.mark.parametrize("ns,nf,nt", GPU_CASES)
def test_fp16_within_bound(ns, nf, nt, order):
    from test_gpu_parity import assert_f16_close, f16_input
    flush(f"[sub-tiles] fp16 ns={ns} nf={nf} nt={nt} {order}")
    x = f16_input(nt, nf, ns, 72)
    eng = X.Engine(ns, nf, compute=X.XGPU_FLOAT16, order=ORDERS[order])
    eng.correlate(X.DeviceBuffer.from_array(x), nt)
    got = eng.dump(triangular=True)
    assert_f16_close(got, oracle.xengine_f64_f16(x, ns, nf, nt), ns, nf, nt)


@pytest.mark.gpu
def test_batch_mixes_tile_sizes():
    """Jobs that fill square tiles and jobs that do not, in one batch."""
    shapes = [(96, 40, 2048), (256, 24, 1024), (16, 3, 300), (96, 33, 4096)]
    flush(f"[sub-tiles] batch {shapes}")
    items, refs = [], []
    for k, (ns, nf, nt) in enumerate(shapes):
        x = oracle.fill_uniform(nt * nf * ns * 4, 80 + k, -128, 127)
        eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=X.TRIANGULAR_ORDER)
        items.append((eng, X.DeviceBuffer.from_array(x), nt))
        alone = X.Engine(ns, nf, compute=X.XGPU_INT8, order=X.TRIANGULAR_ORDER)
        alone.set_tuning(kernel=1)
        alone.correlate(items[-1][1], nt)
        refs.append(alone.dump())
    for _ in range(2):
        X.correlate_batch(items)
    for (eng, _, _), ref in zip(items, refs):
        assert np.array_equal(eng.dump(), 2 * ref)
