"""Time-swizzled int8 blocks read by the real-Gram DMA kernels as they are (the
default tuning): a memory row holds 4 samples, byte e of sample t in byte
4 e + t % 4.

CPU: a model of both kernels' loads and operand reads stays inside the block
and gives every lane its real row's samples.  GPU: results equal the integer
oracle's, and the converted path's (an explicit tuning), exactly.
"""
import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush

ORDERS = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER,
          "tri": X.TRIANGULAR_ORDER}
LANES = np.arange(64)


def chunk_of(slot, row):
    return slot ^ ((row & 4) << 1)


def lds_kstep(block, ts, f, blk, per_tile, nt, t0, ninput):
    """One kstep (32 samples) of one tile side in LDS: 8 memory rows of 8 * per_tile bytes."""
    row_len = 8 * per_tile
    lds = np.full(8 * row_len, 77, np.int8)
    nbytes = min(row_len, (ninput - blk * per_tile) * 8)
    base = (f * ninput + blk * per_tile) * 8 + t0 * ts
    rows = min(max(nt - t0, 0), 32)
    nrec = rows * ts - 4 * ts + nbytes if rows > 0 else 0
    chunks = row_len // 16
    for dma in range(8 * row_len // 1024):
        row = dma * (1024 // row_len) + LANES // chunks
        chunk = chunk_of(LANES % chunks, row)
        voff = np.where(16 * chunk < nbytes, row * 4 * ts + 16 * chunk, 0x7fffff00)
        for lane in LANES:
            at = dma * 1024 + 16 * lane
            if voff[lane] < nrec:
                assert voff[lane] + 16 <= nrec and base + nrec <= nt * ts
                lds[at:at + 16] = block[base + voff[lane]:base + voff[lane] + 16]
            else:
                lds[at:at + 16] = 0
    return lds


@pytest.mark.parametrize("per_tile", [128, 64])      # square tiles, sub-tiles
@pytest.mark.parametrize("ns,nf,nt", [(2, 2, 4), (34, 2, 36), (66, 1, 32), (130, 2, 60)])
def test_loads_and_operands(ns, nf, nt, per_tile):
    ninput, ts, row_len = 2 * ns, nf * ns * 4, 8 * per_tile
    x = oracle.fill_uniform(nt * ts, 61, -128, 127)
    plain = x.reshape(nt, nf, 2 * ninput)
    block = oracle.swizzle(x, ns, nf, nt).reshape(-1)
    for f in range(nf):
        for blk in range((ninput + per_tile - 1) // per_tile):
            for t0 in range(0, nt + 32, 32):
                lds = lds_kstep(block, ts, f, blk, per_tile, nt, t0, ninput)
                for b in range(per_tile // 16):      # 32-real-row blocks
                    kg, r = LANES >> 5, LANES & 31
                    off = kg * 4 * row_len + ((128 * b + 4 * r) ^ (kg << 7))
                    assert len(set((off // 4) % 64)) == 64          # all banks once
                    for lane in LANES:
                        got = np.concatenate([lds[off[lane] + row_len * d:][:4] for d in range(4)])
                        e = blk * 2 * per_tile + 32 * b + r[lane]
                        want = np.zeros(16, np.int8)
                        t = t0 + 16 * kg[lane]
                        if e < 2 * ninput and t < nt:
                            want[:min(16, nt - t)] = plain[t:t + 16, f, e]
                        assert np.array_equal(got, want), (blk, t0, b, lane)


@pytest.mark.gpu
@pytest.mark.parametrize("ns,nf,nt,order", [(2, 1, 4, "tri"), (6, 3, 36, "realimag"), (34, 1, 128, "tri"),
                                            (64, 8, 2048, "regtile"), (66, 5, 500, "realimag"),
                                            (130, 3, 96, "tri"), (202, 37, 60, "realimag"),
                                            (256, 16, 1024, "regtile"), (352, 29, 64, "tri")])
def test_swizzled_exact(ns, nf, nt, order):
    flush(f"[swizzled] ns={ns} nf={nf} nt={nt} {order}")
    per = nt * nf * ns * 4
    x = oracle.fill_uniform(2 * per, 62, -128, 127)
    xs = np.concatenate([oracle.swizzle(x[k * per:(k + 1) * per], ns, nf, nt).reshape(-1) for k in range(2)])
    buf = X.DeviceBuffer.from_array(xs)
    engs = [X.Engine(ns, nf, compute=X.XGPU_INT8, order=ORDERS[order], time_swizzle=4) for _ in range(2)]
    engs[1].set_tuning(kernel=2, staging=2, stage=32)        # converted first
    want = 0
    for k in range(2):
        want = want + oracle.xengine_i64(x[k * per:(k + 1) * per], ns, nf, nt)
        for eng in engs:
            eng.correlate(buf.ptr + k * per, nt)
            assert np.array_equal(eng.dump(wide=True, triangular=True), want)


@pytest.mark.gpu
def test_swizzled_past_the_bound_and_refusals():
    """A block cut at the 32-bit bound is cut between groups of 4 samples; sample
    counts and addresses that were refused still are."""
    ns, nf, nt = 8, 2, 70000
    flush("[swizzled] past the bound")
    x = oracle.fill_uniform(nt * nf * ns * 4, 63, -128, 127)
    buf = X.DeviceBuffer.from_array(oracle.swizzle(x, ns, nf, nt))
    eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=X.TRIANGULAR_ORDER, time_swizzle=4)
    ref = oracle.xengine_i64(x, ns, nf, nt)
    for k in range(1, 4):
        eng.correlate(buf, nt)
        assert np.array_equal(eng.dump(wide=True), k * ref)
    with pytest.raises(X.XgpuError):
        eng.correlate(buf, 6)
    with pytest.raises(X.XgpuError):
        eng.correlate(buf.ptr + 8, 4)
