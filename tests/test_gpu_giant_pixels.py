"""Pixels that blocks rank (csrc/pixel_sort.h rank_block: more than 4096 galaxies, 1024 own galaxies per
block): at the limit and one to either side, at whole and ragged numbers of own sets, two giant pixels
side by side in one block, far beyond, with tied radii, weights and radii that are not numbers apart.
FP64 delta maps follow (r, input order) inside a pixel: bit-exact against the oracle.  Folded and
mixed calls: the same from call to call, whatever order the galaxies arrive in, and within the tests'
bounds of the oracle's and the FP64 path's."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (theta, phi) of three pixels that follow one another at nside 2 (a ring of 8), and one far away
SPOTS = [(1.35, 0.4), (1.35, 1.2), (1.35, 2.0), (2.6, 4.0)]


def catalogue(rng, n, crowds):
    th, ph = np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)
    a = 0
    for (t, p), c in zip(SPOTS, crowds):
        th[a:a + c], ph[a:a + c] = t, p
        a += c
    r = rng.uniform(500.0, 1000.0, n)
    r[::3] = np.round(r[::3])
    q = rng.permutation(n)
    return np.stack([r[q], th[q], ph[q]])


def oracle_modes(am):
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    return om


CROWDS = [(2, (4096,)), (2, (4097,)), (2, (5120,)), (2, (5121, 4097)), (2, (4300, 4097, 9000)), (4, (30001, 5000, 60, 4500)),
          (1, (4200, 4200))]


@pytest.mark.parametrize("nside,crowds", CROWDS)
def test_order_against_the_oracle(nside, crowds):
    n = 700 + sum(crowds)
    print("giant pixels", nside, crowds, flush=True)
    am = S.AnlmModes.from_nl(2, 2, 500.0, 1000.0, nside=nside)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(n)
    cat = catalogue(rng, n, crowds)
    w = rng.uniform(0.5, 1.5, n)
    ref = O.delta_map(oracle_modes(am), cat, 1e-6, 1, win.mask, win.w_ln.reshape(-1, order="F"), w, 4)
    plan = S.Plan(am)
    for _ in range(2):
        assert np.array_equal(plan.delta_map(cat, 1e-6, win, w, 4), ref)


@pytest.mark.parametrize("nside,crowds", CROWDS[:5])
def test_folded_and_mixed_calls(nside, crowds):
    """nside 16 beside the listed spots: galaxies of both hemispheres share folded pixels."""
    n = 4000 + sum(crowds)
    print("giant pixels, calls", nside, crowds, flush=True)
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(n + 1)
    cat = catalogue(rng, n, crowds)
    south = rng.random(n) < 0.3  # some of the giant pixels' galaxies in the mirror pixel
    cat[1, south], cat[2, south] = np.pi - cat[1, south], (cat[2, south] + np.pi) % (2 * np.pi)
    w = rng.uniform(0.5, 1.5, n)
    nbar = n / (4 * np.pi / 3 * (1000.0 ** 3 - 500.0 ** 3))
    ref = O.cat2amln(oracle_modes(am), cat, nbar, 1, win.mask, win.w_ln.reshape(-1, order="F"), w)
    fp64, mixed = S.Plan(am), S.Plan(am, precision="mixed")
    a, m = fp64.cat2amln(cat, nbar, win, w), mixed.cat2amln(cat, nbar, win, w)
    assert np.max(np.abs(a - ref)) <= 1e-10 * np.max(np.abs(ref))
    assert np.max(np.abs(m - ref)) <= 1e-6 * np.max(np.abs(ref))
    for _ in range(3):
        assert np.array_equal(fp64.cat2amln(cat, nbar, win, w), a)
        assert np.array_equal(mixed.cat2amln(cat, nbar, win, w), m)


def test_radii_that_are_not_numbers():
    """Sort keys of NaN and infinite radii in a giant pixel: every galaxy keeps a place of its own (the
    call reports the non-finite result as ever)."""
    print("giant pixel with NaN", flush=True)
    am = S.AnlmModes.from_nl(2, 2, 500.0, 1000.0, nside=2)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(3)
    cat = catalogue(rng, 6000, (5000,))
    cat[0, :4] = np.nan, -np.nan, np.inf, -np.inf
    plan = S.Plan(am)
    with pytest.raises(AssertionError):
        plan.cat2amln(cat, 1e-5, win)
    cat[0, :2] = 0.0
    ref = O.delta_map(oracle_modes(am), cat, 1e-6, 1, win.mask, win.w_ln.reshape(-1, order="F"), None, 4)
    assert np.array_equal(plan.delta_map(cat, 1e-6, win, None, 4), ref)
