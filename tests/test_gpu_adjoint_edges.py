"""The folded adjoint's gather (csrc/fold_kernels.h k_vjp_fold) at its own edges: blocks of 2048 (FP64)
and 4096 (mixed) galaxies, radii on the edges of the radius bins that the case gets, table lengths
that give many bins, and catalogues small enough that their size caps the bins.  Against the
unfolded path; tolerances as for the folded adjoint elsewhere (FP64 1e-11 of the RMS: the rounding of
t; mixed 3e-6: FP32 records, products and ring transforms)."""
import numpy as np
import pytest

import sfb_amd as S

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-11, "mixed": 3e-6}


def bins(am, precision, n):
    """The number of radius bins of a call (at most 7 KB of a map's records each)."""
    table = (16 if precision == "mixed" else 32) * (int(np.diff(am.knot_off).max()) + 1)
    npf = 6 * am.nside ** 2 + 2 * am.nside
    return max(1, min(16, 4 * n // npf, -(-table // (7 << 10))))


def check(am, precision, cat, w, monkeypatch):
    rng = np.random.default_rng(3)
    monkeypatch.setenv("SFB_SEG_SEARCH", "1")
    ref_plan = S.Plan(am, precision=precision)
    monkeypatch.delenv("SFB_SEG_SEARCH")
    plan = S.Plan(am, precision=precision)
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    got, ref = plan.cat2amln_vjp(cat, 1e-5, c, w), ref_plan.cat2amln_vjp(cat, 1e-5, c, w)
    for g, r in zip(got[:2], ref[:2]):
        assert np.max(np.abs(g - r)) <= TOL[precision] * np.sqrt(np.mean(r ** 2))


def sky(rng, r):
    n = r.size
    return np.stack([r, np.arccos(rng.uniform(-1, 1, n)), rng.uniform(0, 2 * np.pi, n)])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [2047, 2048, 2049, 4095, 4096, 4097])
def test_block_edges(n, precision, monkeypatch):
    print("adjoint block edge", n, precision, flush=True)
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    rng = np.random.default_rng(n)
    check(am, precision, sky(rng, rng.uniform(500.0, 1000.0, n)), rng.uniform(0.5, 1.5, n), monkeypatch)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [3103, 6209, 40007])
def test_bin_edges(n, precision, monkeypatch):
    am = S.AnlmModes.from_nl(40, 20, 500.0, 1500.0, nside=32)
    nbin = bins(am, precision, n)
    print("adjoint bin edges", n, precision, nbin, flush=True)
    assert nbin == {3103: 1, 6209: 4}.get(n, nbin) and (n < 40007 or nbin >= 6)
    rng = np.random.default_rng(n)
    edge = 500.0 + 1000.0 * rng.integers(0, nbin + 1, n) / nbin
    r = np.where(rng.random(n) < 0.3, rng.uniform(495.0, 1505.0, n), np.nextafter(edge, rng.choice([0.0, 1e4], n)))
    r[::5] = edge[::5]
    check(am, precision, sky(rng, r), rng.uniform(0.5, 1.5, n), monkeypatch)
