"""The mixed path over the common radial basis (csrc/radial.cpp, csrc/shells.h) against the FP64
path, which is pinned to the oracle: every (n, l) block to 1e-6 of its RMS.  The representation
is held to 6e-8 of a spline's largest value at plan creation, and a block's RMS is at least
a few tenths of the shot noise of the same values, so 1e-6 leaves a factor of a few; catalogues
whose galaxies all sit where the splines are hardest to represent are the edge of that.
Tables that the basis does not represent keep the per-map path."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window, shell_volume, uniform_shell_catalog

pytestmark = pytest.mark.gpu


def block_error(a, ref, am):
    worst, i = 0.0, 0
    for n in range(am.nmax):
        for l in range(int(am.lmax_n[n]) + 1):
            s = slice(i, i + l + 1)
            rms = np.sqrt(np.mean(np.abs(ref[s]) ** 2))
            worst = max(worst, float(np.max(np.abs(a[s] - ref[s])) / rms))
            i += l + 1
    return worst


def both(am, cat, nbar, win, w=None):
    return (S.Plan(am, precision=p).cat2amln(cat, nbar, win, w) for p in ("mixed", "fp64"))


@pytest.mark.parametrize("where", ["lower end", "upper end", "outside", "knots", "few"])
def test_edge_radii(where):
    print("shells", where, flush=True)
    am = S.AnlmModes(0.04, 500.0, 1000.0, nside=32)
    win, _ = separable_unit_window(S, am)
    rng = np.random.default_rng(len(where))
    n = 37 if where == "few" else 30011
    cat = uniform_shell_catalog(n, 500.0, 1000.0, seed=3)
    if where == "lower end":
        cat[0] = 500.0 + 8.0 * rng.random(n) ** 3
    elif where == "upper end":
        cat[0] = 1000.0 - 8.0 * rng.random(n) ** 3
    elif where == "outside":
        cat[0, ::2] = rng.choice([0.0, -1.0, 499.0, 1001.0, 1e30, np.inf, -np.inf], cat[0, ::2].size)
    elif where == "knots":
        q = am.nmaps - 1
        cat[0] = rng.choice(am.knot_x[am.knot_off[q]:am.knot_off[q + 1]], n)
    w = rng.uniform(0.5, 1.5, n)
    for weights in (None, w):
        a, ref = both(am, cat, n / shell_volume(500.0, 1000.0), win, weights)
        e = block_error(a, ref, am)
        print("  worst block", e, flush=True)
        assert e <= 1e-6


@pytest.mark.parametrize("nside,nl", [(2, (20, 8)), (4, (30, 4)), (16, (12, 13))])
def test_small_grids_and_masks(nside, nl):
    """Pixel counts that do not fill a tile, an empty catalogue, a mask with zeros."""
    print("shells grid", nside, nl, flush=True)
    am = S.AnlmModes.from_nl(nl[0], nl[1], 500.0, 1000.0, nside=nside)
    base, _ = separable_unit_window(S, am)
    rng = np.random.default_rng(nside)
    win = S.SeparableArray((rng.random(12 * nside ** 2) < 0.7) * 1.0, base.w_ln, "mask", "w_ln")
    for n in (0, 1, 4001):
        cat = uniform_shell_catalog(n, 500.0, 1000.0, seed=n) if n else np.zeros((3, 0))
        a, ref = both(am, cat, 1e-6, win)
        assert np.max(np.abs(a - ref)) <= 1e-6 * np.sqrt(np.mean(np.abs(ref) ** 2))


def test_unrepresented_tables_keep_the_per_map_path():
    """Knots three times as wide: the splines' own error is 80 times larger than the basis is
    allowed to leave out.  The mixed result still follows these splines."""
    am = S.AnlmModes(0.04, 500.0, 1000.0, nside=16)
    off, xs, ys, ypps = [0], [], [], []
    for n in range(1, am.nmax + 1):
        for l in range(int(am.lmax_n[n - 1]) + 1):
            sp = am.basisfunctions.spline(n, l)
            k = (sp.x.size + 2) // 3
            x = np.linspace(500.0, 1000.0, k)
            c = S.Spline1D(x, sp(x))
            xs.append(c.x), ys.append(c.y), ypps.append(c.ypp)
            off.append(off[-1] + k)
    coarse = S.AnlmModes.from_tables(500.0, 1000.0, 16, am.lmax_n, np.array(off), np.concatenate(xs),
                                     np.concatenate(ys), np.concatenate(ypps))
    win = S.SeparableArray(np.ones(12 * 256), np.nan_to_num(separable_unit_window(S, am)[0].w_ln), "mask", "w_ln")
    cat = uniform_shell_catalog(20000, 500.0, 1000.0, seed=8)
    a, ref = both(coarse, cat, 20000 / shell_volume(500.0, 1000.0), win)
    e = block_error(a, ref, coarse)
    print("coarse tables, worst block", e, flush=True)
    assert e <= 1e-6
