"""What only the mixed precisions use (radial basis, FP32 tile search) is laid out when a plan first
takes one of them: an FP64 plan pays for neither, a plan switched later equals one created so, a
switch that fails leaves the plan as it was, and no phase time is charged to the search."""
import os

import numpy as np
import pytest

import sfb_amd as S
from helpers import separable_unit_window, shell_volume, uniform_shell_catalog
from sfb_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    am = S.AnlmModes(0.05, 500.0, 1000.0, nside=32)
    win, _ = separable_unit_window(S, am, nr=100)
    cat = uniform_shell_catalog(20000, 500.0, 1000.0, seed=4)
    return am, win, cat, 20000 / shell_volume(500.0, 1000.0)


@pytest.mark.parametrize("precision", ["mixed", "bf16x3"])
def test_switched_plan_equals_created_plan(setup, precision):
    am, win, cat, nbar = setup
    plan = S.Plan(am)
    fp64 = plan.cat2amln(cat, nbar, win)
    plan.profile(True)
    plan.set_precision(precision)
    assert all(n == 0 for _, n in plan.phase_times()[0].values())
    plan.profile(False)
    created = S.Plan(am, precision=precision)
    for rep in range(2):
        print("late precision", precision, rep, flush=True)
        assert np.array_equal(plan.cat2amln(cat, nbar, win), created.cat2amln(cat, nbar, win))
        plan.set_precision("fp64")
        assert np.array_equal(plan.cat2amln(cat, nbar, win), fp64)
        plan.set_precision(precision)


def test_failed_switch_keeps_the_plan(setup, monkeypatch):
    am, win, cat, nbar = setup
    plan = S.Plan(am)
    fp64 = plan.cat2amln(cat, nbar, win)
    monkeypatch.setenv("SFB_FAULT", "alloc")
    with pytest.raises(S.SFBError) as e:
        plan.set_precision("mixed")
    assert e.value.code == L.SFB_ERR_DEVICE
    os.environ.pop("SFB_FAULT")
    assert np.array_equal(plan.cat2amln(cat, nbar, win), fp64)
    plan.set_precision("mixed")
    assert np.array_equal(plan.cat2amln(cat, nbar, win), S.Plan(am, precision="mixed").cat2amln(cat, nbar, win))
