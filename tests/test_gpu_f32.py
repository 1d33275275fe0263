"""FP32 engines (int8 input, float visibilities) on the int8 matrix kernels:
results are the plain SIMT kernel's (tuning kernel 1) bit for bit, whichever
tile size or output order runs.  Tiles whose sums may have passed 2^24 are
replaced by that kernel's; it also runs long blocks that add to an integration
and blocks past the int32 bound."""
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


def loud(x, ns, nf, nt, stations):
    """Quiet bytes (+-7), full-range in the given stations."""
    v = x.reshape(nt, nf, ns, 4)
    keep = np.zeros(ns, bool)
    keep[list(stations)] = True
    return np.where(keep[None, None, :, None], v, v % 8).astype(np.int8).reshape(-1)


# sub-tiles, slices, square tiles, partial tiles; sums far past 2^24 everywhere, in
# the last tiles only, nowhere; a second call adds
@pytest.mark.parametrize("order", ["regtile", "realimag", "tri"])
@pytest.mark.parametrize("ns,nf,nt", [(4, 1, 3), (20, 2, 513), (64, 2, 6000), (160, 8, 1500),
                                      (260, 5, 700)])
def test_bit_identical_to_the_plain_kernel(ns, nf, nt, order):
    flush(f"[f32] ns={ns} nf={nf} nt={nt} {order}")
    x = oracle.fill_uniform(2 * nt * nf * ns * 4, 91, -128, 127).reshape(2, -1)
    for stations in (range(ns), [ns - 1], []):
        y = [loud(b, ns, nf, nt, stations) for b in x]
        for blocks in (y[:1], y):
            got, want = run(ns, nf, blocks, order, nt), run(ns, nf, blocks, order, nt, kernel=1)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (len(stations), len(blocks))
    quiet = oracle.xengine_i64(y[0], ns, nf, nt)
    assert np.abs(quiet).max() < 1 << 24
    assert np.array_equal(run(ns, nf, y[:1], order, nt).astype(np.int64), quiet)


def test_graph_and_batch():
    ns, nf, nt = 64, 3, 1500
    flush("[f32] graph, batch")
    x = oracle.fill_uniform(nt * nf * ns * 4, 90, -128, 127)
    want = run(ns, nf, [x], "tri", nt, kernel=1)
    buf = X.DeviceBuffer.from_array(x)
    eng = X.Engine(ns, nf, compute=X.XGPU_FLOAT32, order=X.TRIANGULAR_ORDER)
    eng.set_tuning(graph=1)
    for _ in range(3):
        eng.clear()
        eng.correlate(buf, nt)
        assert np.array_equal(eng.dump(), want)
    eng.clear()
    X.correlate_batch([(eng, buf, nt)])
    assert np.array_equal(eng.dump(), want)


def test_extreme_block_at_the_int32_bound():
    """65535 samples of -128 - 128i fit the integer kernels, 65536 do not: both sums
    are powers of two times integers below 2^24."""
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
