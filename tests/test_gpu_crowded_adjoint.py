"""The adjoint of a catalogue whose galaxies share a few pixels (a pencil beam): the gradients of the
unfolded path, and no time lost to counters that every galaxy adds to (atomics on one address run
one after another: 300 000 galaxies in four pixels took 1.1 to 1.6 ms against 0.3 ms on the whole
sky)."""
import numpy as np
import pytest

import sfb_amd as S

pytestmark = pytest.mark.gpu


def catalogue(n, z, ph, seed):
    rng = np.random.default_rng(seed)
    return np.stack([rng.uniform(500.0, 1000.0, n), np.arccos(rng.uniform(*z, n)), rng.uniform(*ph, n)])


SKY = ((-1.0, 1.0), (0.0, 2 * np.pi))
PENCIL = ((0.485, 0.5), (0.70, 0.715))  # one degree


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 3e-6)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 5003])
def test_gradients(n, precision, tol, monkeypatch):
    """Tolerances as for the folded adjoint (FP64: the rounding of t; mixed: FP32 ring transforms)."""
    print("crowded adjoint", n, precision, flush=True)
    am = S.AnlmModes(0.03, 500.0, 1000.0, nside=16)
    rng = np.random.default_rng(n)
    cat = catalogue(n, *PENCIL, 1)
    w = rng.uniform(0.5, 1.5, n)
    monkeypatch.setenv("SFB_SEG_SEARCH", "1")
    ref_plan = S.Plan(am, precision=precision)
    monkeypatch.delenv("SFB_SEG_SEARCH")
    plan = S.Plan(am, precision=precision)
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    got, ref = plan.cat2amln_vjp(cat, 1e-5, c, w), ref_plan.cat2amln_vjp(cat, 1e-5, c, w)
    for g, r in zip(got[:2], ref[:2]):
        assert np.max(np.abs(g - r)) <= (10 if n == 1 else 1) * tol * np.sqrt(np.mean(r ** 2))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_time(precision):
    am = S.AnlmModes(0.06, 500.0, 1000.0, nside=64)
    plan = S.Plan(am, precision=precision)
    n = 300000
    c = np.ones(plan.nlmsize, dtype=complex)
    ms = []
    for sky in (SKY, PENCIL):
        cat = catalogue(n, *sky, 2)
        plan.cat2amln_vjp(cat, 1e-3, c)
        plan.profile(True)
        for _ in range(5):
            plan.cat2amln_vjp(cat, 1e-3, c)
        ms.append(plan.phase_times()[0]["catalog"][0] / 5)
        plan.profile(False)
    print("catalogue stage, whole sky and pencil beam, ms", precision, ms, flush=True)
    assert ms[1] < 4.0 * ms[0]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 3e-6)])
@pytest.mark.parametrize("n", [28 * 640, 28 * 640 + 1])
def test_dense_sky(n, precision, tol, monkeypatch):
    """On either side of 640 galaxies per folded pixel (nside 2: 28): counting kernels in radius bins,
    and the radix sort without bins."""
    print("dense adjoint", n, precision, flush=True)
    am = S.AnlmModes.from_nl(20, 8, 500.0, 1000.0, nside=2)
    rng = np.random.default_rng(n)
    cat = catalogue(n, *SKY, 3)
    w = rng.uniform(0.5, 1.5, n)
    monkeypatch.setenv("SFB_SEG_SEARCH", "1")
    ref_plan = S.Plan(am, precision=precision)
    monkeypatch.delenv("SFB_SEG_SEARCH")
    plan = S.Plan(am, precision=precision)
    c = rng.normal(size=plan.nlmsize) + 1j * rng.normal(size=plan.nlmsize)
    got, ref = plan.cat2amln_vjp(cat, 1e-5, c, w), ref_plan.cat2amln_vjp(cat, 1e-5, c, w)
    for g, r in zip(got[:2], ref[:2]):
        assert np.max(np.abs(g - r)) <= tol * np.sqrt(np.mean(r ** 2))
