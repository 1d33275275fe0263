"""Which kernels a call launches: the host runtime on the CPU fake of the HIP
layer, from its trace log (XGPU_TRACE)."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush

FAKE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "fake")
needs_gcc = pytest.mark.skipif(shutil.which("gcc") is None or shutil.which("make") is None,
                               reason="needs gcc and make")


def launches(tmp_path, scenario, *args):
    """(how, kernel, samples, slices; 0 slices: square tiles) of every X-engine line."""
    b = subprocess.run(["make", "-s", "-C", FAKE, "test_routes"], capture_output=True, text=True,
                       timeout=600)
    assert b.returncode == 0, b.stdout + b.stderr
    log = tmp_path / "trace.log"
    r = subprocess.run([os.path.join(FAKE, "test_routes"), scenario, *args], capture_output=True,
                       text=True, timeout=600, env=dict(os.environ, XGPU_TRACE=str(log),
                                                        ASAN_OPTIONS="detect_leaks=1:abort_on_error=0"))
    assert r.returncode == 0 and f"ok {scenario}" in r.stdout, (r.stdout + r.stderr)[-4000:]
    out = []
    for l in log.read_text().splitlines():
        m = re.search(r" us (\w+) kernel=(\S+) .* nt=(\d+) ", l)
        if m:
            cut = re.search(r"slices=(\d+)", l)
            out.append((m[1], m[2], int(m[3]), (int(cut[1]) if cut else 1) if "sub-tiles=" in l else 0))
    return out


@needs_gcc
def test_tuning_read_and_set_again(tmp_path):
    """4 stations, 6000 samples: slices of sub-tiles by the library's choice (square tiles when
    the tuning names them), before and after the tuning is read and set again."""
    got = [l for l in launches(tmp_path, "tuning", str(tmp_path)) if l[2] == 6000]
    free, square = ("launch", "xg_xengine_rgd<32,8>", 6000, 16), ("launch", "xg_xengine_rgd<32,8>", 6000, 0)
    swizzled = ("launch", "xg_xengine_rgdz<32,8>", 6000, 16)
    assert got == [free, free, square, square,          # read and set
                   swizzled, swizzled, square, square,  # a tuning that names a kernel: converted
                   free, free, square,                  # after the host autotuner, its result elsewhere
                   square, free]                        # cached lines


@needs_gcc
def test_slices_are_summed_by_a_launch_of_their_own(tmp_path):
    got = launches(tmp_path, "slices")
    assert {(k, n, s) for _, k, n, s in got if k != "xg_xengine_mfma<int8>"} == {
        ("xg_xengine_rgd<32,8>", 6001, 16), ("xg_xengine_rgdz<32,8>", 6000, 16),
        ("xg_xengine_rgdf<32,8>", 6000, 16), ("xg_xengine_f32<large>", 6000, 0),
        ("xg_xengine_f32", 6000, 0)}


@needs_gcc
def test_a_replay_logs_every_launch(tmp_path):
    got = [(how, k) for how, k, _, _ in launches(tmp_path, "replay")]
    pair = ["xg_xengine_rgdf<32,8>", "xg_xengine_f32<large>"]
    assert got == [(how, k) for how in ("capture", "replay", "replay") for k in pair]


@needs_gcc
def test_kernel_by_shape(tmp_path):
    plane, square, stores, f32 = "xg_xengine_mfma<int8>", "xg_xengine_rgd<32,8>", "xg_xengine_rgdp<int8>", "xg_xengine_rgdf<32,8>"
    want = [(2, 520, 4, plane, 0, plane, 0), (6, 520, 64, plane, 0, square, 1),
            (6, 520, 130, square, 1, square, 1), (14, 520, 4, square, 1, square, 1),
            (16, 520, 65, square, 1, square, 1), (18, 520, 4, square, 1, square, 1),
            (14, 512, 4, plane, 0, square, 1), (66, 512, 1, plane, 0, stores, 0),
            (74, 512, 1, stores, 0, stores, 0),
            (6, 256, 4, square, 1, square, 1), (6, 520, 4, f32, 1, f32, 1),
            (16, 2, 64, square, 1, square, 1), (64, 8, 200, square, 1, square, 1),
            (256, 10, 8, square, 0, square, 0), (130, 130, 1, stores, 0, stores, 0),
            (130, 45, 257, square, 0, square, 0),
            (16, 2, 64, f32, 1, f32, 1)]
    got = launches(tmp_path, "shapes")
    for ns, nf, nt, k1, s1, k2, s2 in want:
        a, b = got.pop(0), got.pop(0)
        assert (a[1:], b[1:]) == ((k1, nt, s1), (k2, nt, s2)), (ns, nf, nt)
    assert [(k, n) for _, k, n, _ in got[:5]] == [(f32, 513), ("xg_xengine_f32<large>", 513), ("xg_xengine_f32", 513),
                                                  (f32, 512), (f32, 512)]
    assert [l[1] for l in got[5:]] == [plane, square]


# both sides of the line between the complex-plane kernel and sub-tiles; 8-byte aligned blocks
@pytest.mark.gpu
@pytest.mark.parametrize("ns,nf,nt", [(2, 300, 1), (6, 520, 64), (6, 520, 130), (14, 600, 33), (16, 300, 64),
                                      (66, 512, 1), (72, 520, 65)])
def test_small_arrays_exact(ns, nf, nt):
    flush(f"[small arrays] ns={ns} nf={nf} nt={nt}")
    per = nt * nf * ns * 4
    x = oracle.fill_uniform(2 * per, 95, -128, 127)
    for off in (0, 8):
        bufs = [X.DeviceBuffer.from_array(np.concatenate([np.zeros(off, np.int8), b])) for b in (x[:per], x[per:])]
        eng = X.Engine(ns, nf, compute=X.XGPU_INT8, order=X.TRIANGULAR_ORDER)
        for calls in (1, 2):
            eng.correlate(bufs[calls - 1].ptr + off, nt)
            assert np.array_equal(eng.dump().astype(np.int64), oracle.xengine_i64(x[:calls * per], ns, nf, calls * nt))
        eng.clear()
        X.correlate_batch([(eng, bufs[0].ptr + off, nt)])
        assert np.array_equal(eng.dump().astype(np.int64), oracle.xengine_i64(x[:per], ns, nf, nt))


# launches with plain output stores (xg_xengine_rgdp): more tiles than CUs, partial tiles and
# sample tails, up to the longest block
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["int8", "fp32", "swizzled"])
@pytest.mark.parametrize("ns,nf,nt,order", [(128, 90, 36, X.REGISTER_TILE_TRIANGULAR_ORDER),
                                            (132, 50, 256, X.REGISTER_TILE_TRIANGULAR_ORDER),
                                            (202, 30, 4, X.REAL_IMAG_TRIANGULAR_ORDER),
                                            (130, 45, 100, X.REAL_IMAG_TRIANGULAR_ORDER)])
def test_plain_stores_are_the_general_kernels(ns, nf, nt, order, kind):
    flush(f"[plain stores] {kind} ns={ns} nf={nf} nt={nt}")
    per = nt * nf * ns * 4
    x = oracle.fill_uniform(2 * per, 96, -128, 127)
    compute = X.XGPU_FLOAT32 if kind == "fp32" else X.XGPU_INT8
    swz = 4 if kind == "swizzled" else 0
    eng = X.Engine(ns, nf, compute=compute, order=order, time_swizzle=swz)
    ref = X.Engine(ns, nf, compute=compute, order=order)
    ref.set_tuning(kernel=1)
    for b in (x[:per], x[per:]):  # stored, then added to
        plain = X.DeviceBuffer.from_array(b)
        buf = plain
        if swz:
            buf = X.DeviceBuffer(per)
            X.swizzle_input(buf, plain, ns, nf, nt)
        eng.correlate(buf, nt)
        ref.correlate(plain, nt)
        a, b = eng.dump(), ref.dump()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
