"""Batches whose jobs run partly in sub-tiles and partly in square tiles: one
launch (xg_xengine_mix), so a batch that fails has queued nothing.  On the CPU
the fake of the HIP layer with injected faults and the host view of the
schedule; on the GPU the results against the general kernels (tuning kernel 1),
exactly."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle
import xgpu_amd as X
from conftest import flush
from test_schedule import XG_NXCD, XG_TILE, XgLaunch

FAKE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "fake")
needs_gcc = pytest.mark.skipif(shutil.which("gcc") is None or shutil.which("make") is None,
                               reason="needs gcc and make")


def run_fake(scenario, log):
    b = subprocess.run(["make", "-s", "-C", FAKE, "test_batches"], capture_output=True, text=True,
                       timeout=600)
    assert b.returncode == 0, b.stdout + b.stderr
    r = subprocess.run([os.path.join(FAKE, "test_batches"), scenario], capture_output=True, text=True,
                       timeout=600, env=dict(os.environ, XGPU_TRACE=str(log),
                                             ASAN_OPTIONS="detect_leaks=1:abort_on_error=0"))
    assert r.returncode == 0 and f"ok {scenario}" in r.stdout, (r.stdout + r.stderr)[-4000:]
    return log.read_text().splitlines()


@needs_gcc
def test_failed_batch_leaves_nothing_behind(tmp_path):
    lines = [l for l in run_fake("retry", tmp_path / "trace.log") if "jobs=2" in l]
    assert lines and all("kernel=xg_xengine_mix<int8> sub-tile-jobs=1 " in l for l in lines)


@needs_gcc
def test_graph_steps_of_a_batch_are_kept(tmp_path):
    lines = [l.split()[3] for l in run_fake("cycle", tmp_path / "trace.log")]
    assert lines.count("capture") == 6 and lines.count("replay") == 18


@pytest.mark.parametrize("sub,square", [([(32, 5)], [(64, 1)]), ([(30, 70), (2, 9)], [(200, 3), (64, 11)]),
                                        ([(130, 1)], [(128, 40)])])
def test_units_then_tiles_exactly_once(sub, square):
    """jobs: (stations, channels); sub-tile jobs first."""
    lib, L, chan = X.core(), XgLaunch(), 0
    expect = []
    for i, (ns, nf) in enumerate(sub + square):
        J, tile = L.jobs[i], 64 if i < len(sub) else XG_TILE
        J.nstation, J.nfreq, J.ntime, J.chan_base = ns, nf, 64, chan
        J.nblk = (2 * ns + tile - 1) // tile
        J.pair_tiles = 2 | 1 << 8 if i < len(sub) else 0  # the tiling field
        J.tiles_per_chan = J.nblk * (J.nblk + 1) // 2
        chan += nf
        expect += [(i, f, r, c) for f in range(nf) for r in range(J.nblk) for c in range(r + 1)]
    L.njobs, n = len(sub + square), len(sub)
    lib.xg_plan_launch.argtypes = [C.POINTER(XgLaunch), C.c_int, C.c_int]
    lib.xg_plan_launch(C.byref(L), 256, 1)
    tiles = [L.xcd_start[x][L.njobs] - L.xcd_start[x][n] for x in range(XG_NXCD)]
    assert L.wg_per_xcd == min(32, max(tiles))  # the persistent ones only
    lib.xgh_schedule.argtypes = [C.POINTER(XgLaunch), C.c_int, C.c_int] + [C.POINTER(C.c_int)] * 4
    seen = []
    for x in range(XG_NXCD):
        k, v = 0, [C.c_int() for _ in range(4)]
        while lib.xgh_schedule(C.byref(L), x, k, *[C.byref(a) for a in v]):
            job = v[0].value % 16
            assert (job < n) == (k < L.xcd_start[x][n])
            seen.append((job, v[1].value, v[2].value, v[3].value))
            k += 1
        assert k == L.xcd_start[x][L.njobs]
    assert sorted(seen) == sorted(expect)


# few samples and many channels, a tile on one XCD only; ragged tiles of both
# kinds in an order of their own; several rounds of square tiles
@pytest.mark.gpu
@pytest.mark.parametrize("compute", ["int8", "fp32"])
@pytest.mark.parametrize("shapes", [[(64, 1, 3), (32, 1500, 3)],
                                    [(30, 600, 500), (130, 9, 512), (2, 3, 33), (68, 5, 100)],
                                    [(512, 16, 300), (20, 900, 400), (34, 24, 512)]])
def test_results_are_the_general_kernels(shapes, compute):
    flush(f"[mixed batch] {compute} {shapes}")
    ORDERS = (X.REGISTER_TILE_TRIANGULAR_ORDER, X.REAL_IMAG_TRIANGULAR_ORDER, X.TRIANGULAR_ORDER)
    kind = X.XGPU_INT8 if compute == "int8" else X.XGPU_FLOAT32
    for graph in (0, 1):
        items, alone = [], []
        for k, (ns, nf, nt) in enumerate(shapes):
            x = oracle.fill_uniform(nt * nf * ns * 4, 200 + k, -128, 127)
            order = ORDERS[(k + graph) % 3]
            order = X.TRIANGULAR_ORDER if ns % 4 else order
            pair = [X.Engine(ns, nf, compute=kind, order=order) for _ in range(2)]
            pair[1].set_tuning(kernel=1)
            alone.append(pair[1])
            items.append((pair[0], X.DeviceBuffer.from_array(x), nt))
        if graph:
            items[0][0].set_tuning(graph=1)
        for rep in range(2):  # store and add (FP32: past 2^24), then with graphs replays of them
            for (eng, _, _), ref in zip(items, alone):
                eng.clear()
                ref.clear()
            for _ in range(4):
                X.correlate_batch(items)
                for ref, (eng, buf, nt) in zip(alone, items):
                    ref.correlate(buf, nt)
                    assert np.array_equal(eng.dump(), ref.dump()), (graph, rep, eng.nstation)
        for (eng, buf, _), ref in zip(items, alone):
            eng.close()
            ref.close()
            buf.free()
