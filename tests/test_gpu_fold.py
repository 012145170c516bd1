"""FP64 cat2amln on folded hemispheres (csrc/fold.h) against the oracle: grids where the folded
pixels do not tile slices or windows (nside 1 to 16), catalogues on one hemisphere, on the
equator ring and at the poles, windows that differ between the hemispheres (separable and
dense), weights, no refinement and more than the folded operator takes (the unfolded path), and
a crowded pixel (radix sorts).  Tolerance 1e-10 of each block's RMS, as the FP64 parity tests."""
import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def oracle_view(am):
    om = O.OracleModes.__new__(O.OracleModes)
    om.nside, om.lmax, om.nmax, om.lmax_n = am.nside, am.lmax, am.nmax, am.lmax_n
    om.knot_off, om.knot_x, om.knot_y, om.knot_ypp = am.knot_off, am.knot_x, am.knot_y, am.knot_ypp
    return om


def catalogue(rng, n, sky):
    z = {"full": rng.uniform(-1, 1, n), "south": rng.uniform(-1, 0, n), "north": rng.uniform(0, 1, n),
         "equator": rng.uniform(-0.01, 0.01, n), "poles": rng.choice([-1, 1], n) * (1 - 1e-3 * rng.random(n)),
         "crowd": rng.uniform(-1, 1, n)}[sky]
    ph = rng.uniform(0, 2 * np.pi, n)
    if sky == "crowd":
        z[: 2 * n // 3], ph[: 2 * n // 3] = -0.4321, 1.0
    return np.stack([rng.uniform(490, 1010, n), np.arccos(z), ph])


@pytest.mark.parametrize("nside,nl,niter,n,sky,dense", [
    (1, (3, 2), 3, 50, "full", False), (2, (4, 5), 3, 300, "south", False), (4, (5, 9), 3, 1000, "equator", True),
    (8, (4, 10), 0, 999, "north", False), (8, (6, 9), 2, 3001, "poles", True), (16, (6, 18), 3, 2500, "crowd", False),
    (16, (3, 20), 9, 1000, "full", False), (32, (7, 34), 3, 20011, "full", True), (1, (2, 0), 1, 1, "full", True),
])
def test_fp64_against_oracle(nside, nl, niter, n, sky, dense):
    print("fold", nside, nl, niter, n, sky, dense, flush=True)
    am = S.AnlmModes.from_nl(nl[0], nl[1], 500.0, 1000.0, nside=nside)
    rng = np.random.default_rng(nside * 1000 + n)
    base, _ = separable_unit_window(S, am, nr=40)
    npix = 12 * nside ** 2
    wln = np.nan_to_num(base.w_ln)
    win = S.SeparableArray(rng.uniform(0.2, 1.0, npix), wln, "mask", "w_ln")
    if dense:
        win = win.dense() + 0.1 * rng.normal(size=(npix,) + wln.shape)
    cat, w = catalogue(rng, n, sky), rng.uniform(0.5, 1.5, n)
    plan = S.Plan(am, niter=niter)
    for weights in (w, None):
        got = plan.cat2amln(cat, 2e-6, win, weights)
        a, b = (win.reshape(-1, order="F"), None) if dense else (win.mask, wln.reshape(-1, order="F"))
        ref = O.cat2amln(oracle_view(am), cat, 2e-6, 0 if dense else 1, a, b, w=weights, niter=niter)
        i = 0
        for nn in range(am.nmax):
            for l in range(int(am.lmax_n[nn]) + 1):
                s = slice(i, i + l + 1)
                rms = np.sqrt(np.mean(np.abs(ref[s]) ** 2))
                assert np.max(np.abs(got[s] - ref[s])) <= 1e-10 * rms, (nn + 1, l)
                i += l + 1


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 3e-6)])
@pytest.mark.parametrize("nside,n", [(8, 1), (8, 6143), (16, 6145), (32, 30001)])
def test_adjoint_against_the_unfolded_path(nside, n, precision, tol, monkeypatch):
    """Gradients on folded maps against the unfolded gather (SFB_SEG_SEARCH=1), with radii on the
    end knots (whose slopes count), outside them (flat), on inner knots, and southern galaxies;
    n around a block's 6144 galaxies.  FP64 differs by the rounding of t (1e-12 of a value's
    slope), mixed by FP32 rounding in the ring transforms (the adjoint's 1e-6)."""
    print("fold adjoint", nside, n, precision, flush=True)
    am = S.AnlmModes(0.7 * nside / 1000.0, 500.0, 1000.0, nside=nside)
    rng = np.random.default_rng(n)
    cat = catalogue(rng, n, "full")
    edge = np.array([500.0, 1000.0, np.nextafter(500, 0), np.nextafter(1000, 2000), am.knot_x[7], am.knot_x[-3]])
    cat[0, : min(n, 60)] = np.resize(edge, min(n, 60))
    w = rng.uniform(0.5, 1.5, n)
    plan = S.Plan(am, precision=precision)
    monkeypatch.setenv("SFB_SEG_SEARCH", "1")
    ref_plan = S.Plan(am, precision=precision)
    monkeypatch.delenv("SFB_SEG_SEARCH")
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    got, ref = plan.cat2amln_vjp(cat, 1e-5, c, w), ref_plan.cat2amln_vjp(cat, 1e-5, c, w)
    for g, r in zip(got[:2], ref[:2]):
        rms = np.sqrt(np.mean(r ** 2))
        assert np.max(np.abs(g - r)) <= tol * rms * (10 if n == 1 else 1)
    out = (cat[0] < 500.0) | (cat[0] > 1000.0)
    assert np.all(got[0][out] == 0.0)
