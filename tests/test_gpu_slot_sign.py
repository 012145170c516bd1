"""Folded FP64 maps carry a slot's hemisphere in the sign of its radius (csrc/sfb.hip k_sell_fill):
radii where that could go wrong (negative, both zeros, infinite, on and outside the end knots), and
knots that start at 0 or below (there the call takes the unfolded path), on both hemispheres against
the oracle.  Tolerance 1e-10 of each block's RMS, as the other FP64 tests."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("first", [500.0, 0.0, -100.0])
def test_radii(first, weighted):
    print("slot sign", first, weighted, flush=True)
    base = S.AnlmModes.from_nl(4, 10, 500.0, 1000.0, nside=16)
    win = S.SeparableArray(np.ones(12 * 256), np.nan_to_num(separable_unit_window(S, base, nr=40)[0].w_ln), "mask", "w_ln")
    am = S.AnlmModes.from_tables(500.0, 1000.0, 16, base.lmax_n, base.knot_off, base.knot_x + (first - 500.0),
                                 base.knot_y, base.knot_ypp)
    rng = np.random.default_rng(7)
    n = 3001
    r = rng.uniform(first - 20.0, first + 520.0, n)
    edge = [-3.0, -0.0, 0.0, 3.0, first, first + 500.0, np.nextafter(first, -1e9), np.nextafter(first + 500.0, 1e9),
            np.inf, -np.inf, 1e300, -1e300]
    r[:240] = np.resize(edge, 240)
    cat = np.stack([r, np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)])
    w = rng.uniform(0.5, 1.5, n) if weighted else None
    got = S.Plan(am).cat2amln(cat, 1e-5, win, w)
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    ref = O.cat2amln(om, cat, 1e-5, 1, win.mask, win.w_ln.reshape(-1, order="F"), w=w)
    i = 0
    for nn in range(am.nmax):
        for l in range(int(am.lmax_n[nn]) + 1):
            s = slice(i, i + l + 1)
            assert np.max(np.abs(got[s] - ref[s])) <= 1e-10 * np.sqrt(np.mean(np.abs(ref[s]) ** 2)), (nn + 1, l)
            i += l + 1


def test_nan_radius_is_an_error():
    am = S.AnlmModes.from_nl(4, 10, 500.0, 1000.0, nside=16)
    win, _ = separable_unit_window(S, am, nr=40)
    for z in (0.5, -0.5):
        cat = np.stack([np.full(70, 700.0), np.full(70, np.arccos(z)), np.linspace(0, 6, 70)])
        cat[0, 33] = np.nan
        with pytest.raises(AssertionError):
            S.Plan(am).cat2amln(cat, 1e-5, win)
