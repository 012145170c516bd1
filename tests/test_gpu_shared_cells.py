"""Arrival ranks where lanes of a wavefront share a pixel (csrc/pixel_sort.h arrival_rank): one cell for
all, cells in runs of every length, pairs that no probe distance finds, and a last wavefront with idle
lanes.  Each galaxy gets a place of its own: FP64 delta maps bit-exact against the oracle."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pattern", ["one", "runs", "even parity", "few", "ordered"])
@pytest.mark.parametrize("n", [1, 63, 64, 257, 2049])
def test_shared_cells(pattern, n):
    print("shared cells", pattern, n, flush=True)
    nside = 4
    am = S.AnlmModes.from_nl(2, 2, 500.0, 1000.0, nside=nside)
    win, _ = separable_unit_window(S, am, nr=50)
    rng = np.random.default_rng(n)
    i = np.arange(n)
    if pattern == "one":
        pix = np.full(n, 77)
    elif pattern == "runs":
        pix = np.searchsorted(np.cumsum(np.arange(1, 192)), i, side="right") % 192
    elif pattern == "even parity":  # lanes whose numbers differ in two bits or more share, others do not
        odd = np.array([bin(v & 63).count("1") & 1 for v in i])
        pix = np.where(odd == 0, 5, 6 + i % 180)
    elif pattern == "few":
        pix = rng.integers(0, 3, n)
    else:
        pix = np.sort(rng.integers(0, 192, n))
    th, ph = O.pix2ang_ring(nside, pix)
    cat = np.stack([rng.uniform(500.0, 1000.0, n), th, ph])
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    ref = O.delta_map(om, cat, 1e-6, 1, win.mask, win.w_ln.reshape(-1, order="F"), None, 4)
    assert np.array_equal(S.Plan(am).delta_map(cat, 1e-6, win, None, 4), ref)
