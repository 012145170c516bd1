"""The catalogue's grouping by pixel (csrc/pixel_sort.h): counting kernels with a pairwise rank
inside a pixel, and the radix sorts for crowded pixels.  FP64 delta maps are bit-exact against
the oracle, whose sums follow (r, input order) inside a pixel: at the rank's limit of 512
galaxies per pixel and one to either side, far beyond it (the call is redone), above the mean
that goes to the radix sorts at once, with tied radii and with fewer pixels than a scan chunk
or a window of the sliced layout."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _oracle_modes_from(am):
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    return om


def _catalogue(rng, n, crowd):
    th, ph = np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)
    th[:crowd], ph[:crowd] = 1.2345, 2.3456  # one pixel
    r = rng.uniform(500.0, 1000.0, n)
    r[: n // 3] = np.round(r[: n // 3])  # ties
    p = rng.permutation(n)
    return np.stack([r[p], th[p], ph[p]])


@pytest.mark.parametrize("nside,n,crowd", [(1, 1, 1), (2, 700, 0), (4, 900, 511), (4, 900, 512), (8, 2000, 513),
                                           (8, 6000, 5000), (2, 48 * 97, 0), (16, 20000, 300)])
def test_fp64_delta_maps_bitexact(nside, n, crowd):
    print("pixel sort", nside, n, crowd, flush=True)
    am = S.AnlmModes.from_nl(2, 2, 500.0, 1000.0, nside=nside)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(nside + n)
    cat = _catalogue(rng, n, min(crowd, n))
    w = rng.uniform(0.5, 1.5, n)
    plan, om = S.Plan(am), _oracle_modes_from(am)
    for weights in (w, None, w):  # the second and third calls run with what the first left
        got = plan.delta_map(cat, 1e-6, win, weights, 4)
        ref = O.delta_map(om, cat, 1e-6, 1, win.mask, win.w_ln.reshape(-1, order="F"), weights, 4)
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_crowded_pixel_in_a_batch(precision):
    """A mock that crowds a pixel is redone; the others and later calls are as alone."""
    print("crowded batch", precision, flush=True)
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(5)
    cats = [_catalogue(rng, 3000, c) for c in (0, 600, 10)]
    plan = S.Plan(am, precision=precision)
    for graph in (False, True):
        plan.set_batch_graph(graph)
        got = plan.cat2amln_batch(cats, 1e-5, win)
        for c, g in zip(cats, got):
            assert np.array_equal(g, S.Plan(am, precision=precision).cat2amln(c, 1e-5, win))
