"""Which kernels a call launches: the host runtime on the CPU fake of the HIP
layer, from its trace log (XGPU_TRACE)."""
import os
import re
import shutil
import subprocess

import pytest

FAKE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "fake")
pytestmark = pytest.mark.skipif(shutil.which("gcc") is None or shutil.which("make") is None,
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


def test_slices_are_summed_by_a_launch_of_their_own(tmp_path):
    got = launches(tmp_path, "slices")
    assert {(k, n, s) for _, k, n, s in got if k != "xg_xengine_mfma<int8>"} == {
        ("xg_xengine_rgd<32,8>", 6001, 16), ("xg_xengine_rgdz<32,8>", 6000, 16),
        ("xg_xengine_rgdf<32,8>", 6000, 16), ("xg_xengine_f32<large>", 6000, 0),
        ("xg_xengine_f32", 6000, 0)}


def test_a_replay_logs_every_launch(tmp_path):
    got = [(how, k) for how, k, _, _ in launches(tmp_path, "replay")]
    pair = ["xg_xengine_rgdf<32,8>", "xg_xengine_f32<large>"]
    assert got == [(how, k) for how in ("capture", "replay", "replay") for k in pair]
