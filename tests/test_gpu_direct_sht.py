"""map2alm with its refinements as one operator (csrc/sht_direct.h) against the oracle's
pixel-space iteration, at the edges of its rule: no refinement, one, more than it folds (the
iterated form), lmax from 0 to where whole equatorial rings alias, one map and an odd number
of maps; and its transpose (the adjoint's ring side) through the inner product.

Tolerance: both sides are FP64 sums of fewer than 1e4 terms bounded by the largest |a|, so
rounding stays below ~1e4 x 1.1e-16 of it; 1e-12 as for the iterated form."""
import numpy as np
import pytest

import sfb_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside,lmax,niter,nmap", [
    (4, 1, 3, 1), (4, 5, 3, 5), (8, 9, 1, 3), (8, 10, 2, 7), (16, 19, 4, 1), (16, 23, 8, 2),
    (16, 17, 9, 3), (8, 31, 2, 1), (32, 35, 3, 37), (64, 66, 3, 2),
])
def test_map2alm_direct_vs_oracle(nside, lmax, niter, nmap):
    print("map2alm direct", nside, lmax, niter, nmap, flush=True)
    am = S.AnlmModes.from_nl(max(2, -(-nmap // (lmax + 1))), lmax, 500.0, 1000.0, nside=nside)
    plan = S.Plan(am, niter=niter)
    maps = np.random.default_rng(nside * 100 + lmax).normal(size=(nmap, 12 * nside * nside))
    got = plan.map2alm(maps)
    for i in range(0, nmap, max(1, nmap - 1)):
        ref = O.map2alm(nside, lmax, maps[i], niter)
        err = np.max(np.abs(got[i] - ref)) / np.max(np.abs(ref))
        assert err < 1e-12, err


@pytest.mark.parametrize("nside,kmax,niter", [(8, 0.02, 1), (16, 0.022, 3), (16, 0.016, 9)])
def test_adjoint_direct_inner_product(nside, kmax, niter):
    """<c, a(w)> = <dL/dw, w> + <c, a(0)>: a is affine in the weights."""
    print("adjoint direct", nside, kmax, niter, flush=True)
    am = S.AnlmModes(kmax, 500.0, 1000.0, nside=nside)
    plan = S.Plan(am, niter=niter)
    rng = np.random.default_rng(nside)
    N = 999
    cat = np.stack([rng.uniform(500, 1000, N), np.arccos(rng.uniform(-1, 1, N)), rng.uniform(0, 2 * np.pi, N)])
    w = rng.uniform(0.5, 1.5, N)
    win = S.SeparableArray(np.zeros(plan.npix), np.zeros((am.lmax + 1, am.nmax)), "mask", "w_ln")
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    a = plan.cat2amln(cat, 1e-6, win, w)
    _, dw, _ = plan.cat2amln_vjp(cat, 1e-6, c, w)
    lhs = float(np.sum(c.real * a.real + c.imag * a.imag))
    scale = float(np.sum(np.abs(c) * np.abs(a)))
    assert abs(lhs - float(np.dot(dw, w))) <= 1e-12 * scale
