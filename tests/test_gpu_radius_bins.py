"""Adjoint gather on radius bins (csrc/fold_kernels.h k_vjp_fold) against the unfolded path: the
staged radial range of a block where it can go wrong: all radii alike, on the outermost knots, all
outside, two far shells in one block, radii in steps that fall on bin edges, and more maps per
knot group than one stage holds.  Tolerances as for the folded adjoint: 1e-11 of the RMS in FP64
(knots' rounding 1e-13 times the slopes' growth), 3e-6 with FP32 records and products."""
import numpy as np
import pytest

import sfb_amd as S

pytestmark = pytest.mark.gpu

RADII = {
    "alike": lambda rng, n: np.full(n, 731.25),
    "ends": lambda rng, n: rng.choice([500.0, 1000.0], n),
    "outside": lambda rng, n: rng.choice([480.0, 1020.0, 600.0], n, p=[0.45, 0.45, 0.1]),
    "shells": lambda rng, n: np.where(rng.random(n) < 0.5, 510.0, 990.0) + rng.uniform(-2, 2, n),
    "edges": lambda rng, n: 500.0 + 500.0 * rng.integers(0, 17, n) / 16,
}


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 3e-6)])
@pytest.mark.parametrize("kind", sorted(RADII))
def test_adjoint_radii(kind, precision, tol, monkeypatch):
    nside, n = 32, 40007
    am = S.AnlmModes(0.05, 500.0, 1000.0, nside=nside)
    rng = np.random.default_rng(len(kind))
    cat = np.stack([RADII[kind](rng, n), np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)])
    plan = S.Plan(am, precision=precision)
    monkeypatch.setenv("SFB_SEG_SEARCH", "1")
    ref_plan = S.Plan(am, precision="fp64")
    monkeypatch.delenv("SFB_SEG_SEARCH")
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    w = rng.uniform(0.5, 2.0, n)
    got, ref = plan.cat2amln_vjp(cat, 1e-5, c, w), ref_plan.cat2amln_vjp(cat, 1e-5, c, w)
    for g, r in zip(got[:2], ref[:2]):
        rms = np.sqrt(np.mean(np.square(r)))
        assert np.max(np.abs(g - r)) <= tol * max(rms, 1e-300)
