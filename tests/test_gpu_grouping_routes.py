"""Batches whose mocks group their catalogues in different ways (csrc/pixel_sort.h: counting
kernels up to 96 galaxies per pixel on average, 1024 in FP64, radix sorts beyond) and plans that have met a
crowded pixel: every call returns what a plan of its own returns, eager and as a graph, on the
first launch and on the next."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window

pytestmark = pytest.mark.gpu


def catalogue(rng, n, crowd=0):
    th, ph = np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)
    th[:crowd], ph[:crowd] = 1.2345, 2.3456
    p = rng.permutation(n)
    return np.stack([rng.uniform(500.0, 1000.0, n), th, ph])[:, p]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_on_both_sides_of_the_mean(precision, graph):
    """nside 2: 48 pixels, 28 folded; one galaxy beyond the line, on it, and far below in one batch, on
    a fresh plan."""
    am = S.AnlmModes.from_nl(20, 8, 500.0, 1000.0, nside=2)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(11)
    line = 28 * 1024 if precision == "fp64" else 48 * 96
    cats = [catalogue(rng, n) for n in (500, line + 1, 28 * 96, line, 3)]
    alone = [S.Plan(am, precision=precision).cat2amln(c, 1e-5, win) for c in cats]
    plan = S.Plan(am, precision=precision)
    plan.set_batch_graph(graph)
    for rep in range(3):
        print("grouping routes", precision, graph, rep, flush=True)
        got = plan.cat2amln_batch(cats, 1e-5, win)
        assert all(np.array_equal(g, a) for g, a in zip(got, alone))
        plan.cat2amln(cats[0], 1e-5, win)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_crowded_mock_on_a_fresh_plan(precision, graph):
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(12)
    cats = [catalogue(rng, 3000, c) for c in (0, 600, 10)]
    alone = [S.Plan(am, precision=precision).cat2amln(c, 1e-5, win) for c in cats]
    plan = S.Plan(am, precision=precision)
    plan.set_batch_graph(graph)
    for rep in range(3):
        print("crowded batch", precision, graph, rep, flush=True)
        got = plan.cat2amln_batch(cats, 1e-5, win)
        assert all(np.array_equal(g, a) for g, a in zip(got, alone))
        plan.cat2amln(cats[0], 1e-5, win)


@pytest.mark.parametrize("nside,n,crowd", [(4, 3000, 64), (4, 3000, 65), (2, 2500, 320), (4, 6000, 4097),
                                           (16, 60000, 30000), (1, 1100, 300)])
def test_crowded_pixels_in_order(nside, n, crowd):
    """FP64 delta maps follow (r, input order) inside a pixel at the size where wavefronts rank pixel
    by pixel, one beyond, whole multiples of a wavefront and far beyond, several crowded pixels
    in one wavefront, with tied radii: bit-exact against the oracle."""
    from oracle import oracle as O

    print("crowded order", nside, n, crowd, flush=True)
    am = S.AnlmModes.from_nl(2, 2, 500.0, 1000.0, nside=nside)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(n + crowd)
    cat = catalogue(rng, n, crowd)
    cat[0, ::3] = np.round(cat[0, ::3])
    w = rng.uniform(0.5, 1.5, n)
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    ref = O.delta_map(om, cat, 1e-6, 1, win.mask, win.w_ln.reshape(-1, order="F"), w, 4)
    assert np.array_equal(S.Plan(am).delta_map(cat, 1e-6, win, w, 4), ref)


@pytest.mark.parametrize("precision,nl", [("fp64", (3, 2)), ("mixed", (20, 8))])
def test_beyond_the_rank(precision, nl):
    """2^20 + 1 galaxies in one pixel: the call is redone with the radix sorts; the next call is
    what it was before."""
    print("beyond the rank", precision, flush=True)
    am = S.AnlmModes.from_nl(nl[0], nl[1], 500.0, 1000.0, nside=64)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(13)
    big, small = catalogue(rng, (1 << 20) + 2001, (1 << 20) + 1), catalogue(rng, 2000)
    assert big.shape[1] <= 96 * (6 * 64 ** 2 + 128)  # not by its mean
    plan = S.Plan(am, precision=precision)
    before = plan.cat2amln(small, 1e-5, win)
    one = plan.cat2amln(big, 1e-3, win)
    assert np.array_equal(plan.cat2amln(small, 1e-5, win), before)
    # the same sums in another order: 1e6 terms of one size, each pixel's rounding below 1e-10
    other = plan.cat2amln(big[:, rng.permutation(big.shape[1])], 1e-3, win)
    assert np.max(np.abs(other - one)) <= 1e-9 * np.max(np.abs(one))
    got = plan.cat2amln_batch([small, big], [1e-5, 1e-3], win)
    assert np.array_equal(got[0], before) and np.array_equal(got[1], one)
