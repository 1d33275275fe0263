"""FP32 engines (int8 input, float visibilities) on the int8 matrix kernels:
each launch's integer sums are exact and rounded to float once, whichever tile
size or output order runs; the plain SIMT kernel stays behind tuning kernel 1
and serves blocks past the int32 bound."""
import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush

pytestmark = pytest.mark.gpu

ORDERS = {"regtile": X.REGISTER_TILE_TRIANGULAR_ORDER, "realimag": X.REAL_IMAG_TRIANGULAR_ORDER,
          "tri": X.TRIANGULAR_ORDER}


def run(ns, nf, blocks, order, nt, **tuning):
    eng = X.Engine(ns, nf, compute=X.XGPU_FLOAT32, order=ORDERS[order])
    if tuning:
        eng.set_tuning(**tuning)
    for b in blocks:
        eng.correlate(X.DeviceBuffer.from_array(b), nt)
        eng.synchronize()
    return eng.dump(triangular=True)


# sub-tiles, slices, square tiles, partial tiles; sums far past 2^24
@pytest.mark.parametrize("order", ["regtile", "realimag", "tri"])
@pytest.mark.parametrize("ns,nf,nt", [(4, 1, 3), (20, 2, 129), (64, 2, 6000), (160, 8, 1500),
                                      (260, 5, 700)])
def test_sums_rounded_once(ns, nf, nt, order):
    flush(f"[f32] ns={ns} nf={nf} nt={nt} {order}")
    x = oracle.fill_uniform(2 * nt * nf * ns * 4, 91, -128, 127).reshape(2, -1)
    sums = [oracle.xengine_i64(b, ns, nf, nt).astype(np.float32) for b in x]
    assert np.array_equal(run(ns, nf, x[:1], order, nt), sums[0])
    assert np.array_equal(run(ns, nf, x, order, nt), sums[0] + sums[1])  # a second call adds


def test_extreme_block_at_the_int32_bound():
    """65535 samples of -128 - 128i run on the integer kernels; 65536 do not fit int32
    and run on the SIMT kernel: both sums are powers of two times integers below 2^24."""
    ns, nf = 4, 1
    for nt in (65535, 65536):
        flush(f"[f32] bound nt={nt}")
        got = run(ns, nf, [np.full(nt * nf * ns * 4, -128, dtype=np.int8)], "tri", nt)
        v = got.reshape(-1, 2)
        assert np.all(v[:, 0] == np.float32(nt * 2 * 128 * 128)) and np.all(v[:, 1] == 0)


def test_plain_kernel_agrees_below_2_24():
    ns, nf, nt = 96, 3, 400
    x = oracle.fill_uniform(nt * nf * ns * 4, 92, -128, 127)
    flush("[f32] plain kernel")
    assert np.array_equal(run(ns, nf, [x], "regtile", nt), run(ns, nf, [x], "regtile", nt, kernel=1))
