"""The host fit of the mixed path's radial basis (csrc/radial.cpp) on its own, on the CPU: an allocation
that fails at any point, those for its threads included, gives `no basis` and never ends the
process; tables without knots are turned down before anything is read; and bench.py's count of
the basis functions is the one the fit makes."""
import os
import subprocess
import sys

import numpy as np
import pytest

import sfb_amd as S

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "sphericalfourierbesseldecompositions.jl_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("radial") / "driver")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-pthread", "-I", CSRC, os.path.join(HERE, "radial_driver.cpp"),
                           os.path.join(CSRC, "radial.cpp"), "-o", exe])

    def run(*args):
        return subprocess.run([exe, *args], capture_output=True, text=True, timeout=60)

    return run


def table(path, am, maps=None):
    n = am.nmaps if maps is None else maps
    off = np.asarray(am.knot_off[:n + 1], dtype=np.int64)
    with open(path, "wb") as f:
        np.array([n, off[-1]], dtype=np.int64).tofile(f)
        off.tofile(f)
        for a in (am.knot_x, am.knot_y, am.knot_ypp):
            np.asarray(a[:off[-1]], dtype=np.float64).tofile(f)
    return str(path)


def test_allocation_failures(driver, tmp_path):
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    r = driver("fail", table(tmp_path / "t", am))
    assert r.returncode == 0, (r.returncode, r.stderr[-300:])
    tried, ok, nc = map(int, r.stdout.split())
    assert tried > 10 and ok == 1 and nc > 20


def test_tables_without_knots(driver):
    r = driver("empty")
    assert r.returncode == 0, r.returncode
    assert r.stdout.split() == ["0", "0"]


@pytest.mark.parametrize("kmax,rmin,rmax,nside", [(0.03, 500.0, 1000.0, 16), (0.05, 500.0, 1000.0, 32),
                                                  (0.1, 500.0, 1500.0, 128)])
def test_bench_counts_the_same_functions(driver, tmp_path, kmax, rmin, rmax, nside):
    sys.path.insert(0, ROOT)
    import bench

    am = S.AnlmModes(kmax, rmin, rmax, nside=nside)
    # (the finest table sets the breaks; the others only have to share its ends)
    q = int(np.argmax(np.diff(am.knot_off)))
    lo, hi = am.knot_off[q], am.knot_off[q + 1]
    with open(tmp_path / "t", "wb") as f:
        np.array([1, hi - lo, 0, hi - lo], dtype=np.int64).tofile(f)
        for a in (am.knot_x, am.knot_y, am.knot_ypp):
            np.asarray(a[lo:hi], dtype=np.float64).tofile(f)
    r = driver("count", str(tmp_path / "t"))
    assert r.returncode == 0
    ok, nc = map(int, r.stdout.split())
    assert ok == 1 and nc == bench.shell_count(am)
