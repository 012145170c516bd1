"""Mixed calls with many galaxies per pixel on small grids (csrc/shells.h shell_parts): the spread of a
block's galaxies in parts, at sizes where a part begins and ends, against the FP64 path (every (n, l)
block to 1e-6 of its RMS, as the other mixed tests), the same from call to call, and no slower than
the FP64 path's own scatter (4e6 galaxies at nside 16 took 2.9 ms in 192 blocks)."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window, shell_volume, uniform_shell_catalog
from test_gpu_shells import block_error

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside,nl,n", [(2, (20, 8), 3 * 512 - 1), (2, (20, 8), 3 * 512), (2, (20, 8), 60001),
                                        (4, (30, 8), 12 * 1024), (8, (30, 12), 300007), (16, (30, 12), 196608),
                                        (32, (30, 12), 1600001)])
def test_parts(nside, nl, n):
    print("shell parts", nside, nl, n, flush=True)
    am = S.AnlmModes.from_nl(nl[0], nl[1], 500.0, 1000.0, nside=nside)
    base, _ = separable_unit_window(S, am)
    rng = np.random.default_rng(nside)
    win = S.SeparableArray(rng.uniform(0.2, 1.0, 12 * nside ** 2), base.w_ln, "mask", "w_ln")
    cat = uniform_shell_catalog(n, 500.0, 1000.0, seed=n)
    cat[2, : n // 2] *= 0.5  # uneven pixels
    nbar = n / shell_volume(500.0, 1000.0)
    for w in (None, rng.uniform(0.5, 1.5, n)):
        plan = S.Plan(am, precision="mixed")
        a = plan.cat2amln(cat, nbar, win, w)
        e = block_error(a, S.Plan(am).cat2amln(cat, nbar, win, w), am)
        print("  worst block", e, flush=True)
        assert e <= 1e-6
        assert np.array_equal(plan.cat2amln(cat, nbar, win, w), a)


def test_time():
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    win, _ = separable_unit_window(S, am)
    n = 4000000
    cat = uniform_shell_catalog(n, 500.0, 1000.0, seed=1)
    ms = {}
    for prec in ("fp64", "mixed"):
        plan = S.Plan(am, precision=prec)
        plan.cat2amln(cat, n / shell_volume(500.0, 1000.0), win)
        plan.profile(True)
        for _ in range(3):
            plan.cat2amln(cat, n / shell_volume(500.0, 1000.0), win)
        t = plan.phase_times()[0]
        ms[prec] = (t["scatter"][0] + t["segment"][0]) / 3
    print("scatter, ms", ms, flush=True)
    assert ms["mixed"] < ms["fp64"]
