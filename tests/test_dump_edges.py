"""Triangular device dumps at the edges of the reorder kernels' split: cells
in workgroups of 64 or 128 across channels, the row of a cell from a float
square root.

CPU: the root names the row or a neighbour for every row up to the largest
station count, also two units in the last place off.  GPU: dumps equal the
integer oracle's result exactly in every form (register-tile and real/imag
order, narrow and wide, before and after a spill, aligned and one element off).
"""
import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush

ORDERS = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER}


def test_row_of_a_cell_from_a_float_root():
    i = np.arange(32640, dtype=np.uint64)         # the largest station count
    for b in (i * (i + 1) // 2, i * (i + 1) // 2 + i):      # first and last cell of each row
        r = np.sqrt(np.float32(8) * b.astype(np.float32) + np.float32(1))
        for ulp in (-2, 0, 2):
            q = r + np.float32(ulp) * np.spacing(r)
            est = ((q - np.float32(1)) * np.float32(0.5)).astype(np.int64)
            assert np.abs(est - i.astype(np.int64)).max() <= 1 and est.min() >= 0
            est = est.astype(np.uint64)
            assert ((est + 1) * (est + 2) < 1 << 32).all()
            est = np.where(est * (est + 1) // 2 > b, est - 1, est)
            est = np.where((est + 1) * (est + 2) // 2 <= b, est + 1, est)
            assert (est == i).all()


# cells per channel: 3, 10, 66, 78, 136, 595 (> 4 x 128), 132355; of 3 cells, 70001 channels
@pytest.mark.gpu
@pytest.mark.parametrize("ns,nf,order", [(2, 5, "realimag"), (4, 3, "regtile"), (12, 2, "regtile"),
                                         (16, 7, "regtile"), (34, 3, "realimag"), (100, 2, "regtile"),
                                         (514, 1, "realimag"), (516, 2, "regtile"),
                                         (2, 70001, "realimag")])
def test_device_dumps(ns, nf, order):
    flush(f"[dump] ns={ns} nf={nf} {order}")
    nt, big = 2, 70000                            # 2 x 70000 samples pass the spill limit
    x = oracle.fill_uniform(nt * nf * ns * 4, 51, -128, 127)
    eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=ORDERS[order])
    buf = X.DeviceBuffer.from_array(x)
    zero = X.DeviceBuffer(big * nf * ns * 4) if ns * nf < 1000 else None
    if zero:
        zero.fill_uniform_int8(1, 0, 0)
    want = oracle.xengine_i64(x, ns, nf, nt)
    out = X.DeviceBuffer(2 * eng.tri_len * 8 + 16)
    for spilled in (False, True) if zero else (False,):
        eng.correlate(buf, nt)
        if spilled:
            want = 2 * want
            for _ in range(3):
                eng.correlate(zero, big)
        for wide, dt, esz in ((False, np.int32, 4), (True, np.int64, 8)):
            flags = X.XGPU_DUMP_DEVICE | X.XGPU_DUMP_TRIANGULAR | (X.XGPU_DUMP_WIDE if wide else 0)
            for off in (0, esz):
                out.fill_uniform_int8(52 + off, -127, 127)
                X.check(X.core().xgpuAmdDump(eng.handle, out.ptr + off, flags))
                got = out.download(dt, count=2 * eng.tri_len, offset=off)
                assert np.array_equal(got, want.astype(dt)), (spilled, wide, off)
