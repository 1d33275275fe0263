"""Blocks that are not whole 16-byte chunks on the real-Gram DMA kernels: int8
arrays with nstation % 4 == 2 and blocks at 8-byte aligned addresses.  The
global->LDS loads are range-checked per dword, so the last chunk of the block's
last sample is cut at the block's end.

CPU: a model of the square-tile kernels' loads stays inside the block.  GPU:
int8 and FP32 results equal the integer oracle's, fp16 results stay within the
accumulation bound, and equal work on the general kernels (tuning kernel 1).
"""
import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush

ORDERS = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER,
          "tri": X.TRIANGULAR_ORDER}
OOR = 0x7fffff00


@pytest.mark.parametrize("ns,nf,nt", [(2, 1, 1), (6, 3, 33), (66, 1, 40), (130, 2, 65), (202, 3, 31)])
@pytest.mark.parametrize("stg", [32, 64])
def test_square_tile_loads_in_bounds(ns, nf, nt, stg):
    """rgd_tile, int8: per stage and side one resource, 2 (4) DMAs per wave."""
    ts, ninput = nf * ns * 4, 2 * ns
    lanes = np.arange(64)
    srow, slot = lanes // 16, lanes % 16
    nblk = (ninput + 127) // 128
    for f in {0, nf - 1}:
        for rb in range(nblk):
            for cb in range(rb + 1):
                for side, blk in ((0, rb), (1, cb)):
                    if side and rb == cb:
                        continue  # every lane is out of range
                    nbytes = 256 if side else min(256, (ninput - rb * 128) * 2)
                    assert nbytes <= (ninput - blk * 128) * 2
                    for st in range((nt + stg - 1) // stg + 8):
                        rows = max(min(nt - st * stg, stg), 0)
                        base = f * ninput * 2 + blk * 256 + st * stg * ts
                        nrec = rows * ts - ts + nbytes if rows > 0 else 0
                        got = np.zeros((stg, 16), int)
                        for wave in range(4):
                            x = slot ^ ((wave * 4 + srow) & 7)
                            chunk = x ^ ((x & 1) << 3)
                            for j in range(stg // 16):
                                row = (4 * j + wave) * 4 + srow
                                voff = np.where(blk * 128 + 8 * chunk < ninput, row * ts + 16 * chunk, OOR)
                                ok = voff < nrec
                                end = np.minimum(base + voff[ok] + 16, base + nrec)
                                assert (end <= nt * ts).all()
                                np.add.at(got, (row[ok], chunk[ok]), 1)
                        assert (got[:rows, :(nbytes + 15) // 16] == 1).all()
                        assert (got[rows:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("compute", [X.XGPU_INT8, X.XGPU_FLOAT32])
@pytest.mark.parametrize("stage", [0, 32, 64])   # 0: the library's choice of tiles
@pytest.mark.parametrize("ns,nf,nt,order", [(2, 1, 5, "tri"), (6, 3, 33, "realimag"),
                                            (34, 1, 129, "tri"), (66, 5, 257, "realimag"),
                                            (130, 3, 95, "tri"), (202, 3, 501, "realimag"),
                                            (100, 1, 77, "regtile")])
def test_odd_groups_exact(ns, nf, nt, order, stage, compute):
    flush(f"[unaligned] compute={compute} ns={ns} nf={nf} nt={nt} {order} stage={stage}")
    per = nt * nf * ns * 4
    x = oracle.fill_uniform(2 * per, 93, -128, 127)
    buf = X.DeviceBuffer(2 * per + 8)      # blocks at 8 mod 16, or 16 when a block is odd
    buf.upload(x, 8)
    eng = X.Engine(ns, nf, compute=compute, order=ORDERS[order])
    if stage:
        eng.set_tuning(kernel=2, staging=2, stage=stage)
    want = 0
    for k in range(2):
        eng.correlate(buf.ptr + 8 + k * per, nt)
        want = want + oracle.xengine_i64(x[k * per:(k + 1) * per], ns, nf, nt)
        assert np.abs(want).max() < 1 << 24        # exact in float too
        assert np.array_equal(eng.dump(wide=True, triangular=True), want.astype(eng.wide_dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [0, 16, 32])
@pytest.mark.parametrize("ns,nf,nt", [(6, 3, 33), (66, 2, 130), (130, 1, 70)])
def test_fp16_at_8_byte_alignment(ns, nf, nt, stage):
    from test_gpu_parity import assert_f16_close, f16_input
    flush(f"[unaligned] fp16 ns={ns} nf={nf} nt={nt} stage={stage}")
    x = f16_input(nt, nf, ns, 94)
    buf = X.DeviceBuffer(x.nbytes + 8)
    buf.upload(x, 8)
    eng = X.Engine(ns, nf, compute=X.XGPU_FLOAT16, order=X.TRIANGULAR_ORDER)
    if stage:
        eng.set_tuning(kernel=2, staging=2, stage=stage)
    eng.correlate(buf.ptr + 8, nt)
    assert_f16_close(eng.dump(), oracle.xengine_f64_f16(x, ns, nf, nt), ns, nf, nt)


@pytest.mark.gpu
def test_batch_keeps_to_the_first_engines_kernel():
    """A register-staged first engine cannot take an unaligned second job: the
    whole batch runs on the general kernel, exactly."""
    shapes = [(64, 3, 200), (34, 2, 130)]
    flush("[unaligned] batch")
    items, refs = [], []
    for k, (ns, nf, nt) in enumerate(shapes):
        x = oracle.fill_uniform(nt * nf * ns * 4, 95 + k, -128, 127)
        eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=X.TRIANGULAR_ORDER)
        if k == 0:
            eng.set_tuning(kernel=2, staging=1, stage=64)
        items.append((eng, X.DeviceBuffer.from_array(x), nt))
        refs.append(oracle.xengine_i64(x, ns, nf, nt))
    X.correlate_batch(items)
    for (eng, _, _), ref in zip(items, refs):
        assert np.array_equal(eng.dump(wide=True), ref)
