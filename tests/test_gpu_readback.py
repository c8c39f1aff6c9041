"""Residual histories longer than one batch of the pinned collection buffer
(32 steps): the same bits as steps asked for one at a time, for a single case
and for harmonic balance with one and with several solver cycles; and field
read-backs of any subset."""
import ctypes
import dataclasses

import numpy as np
import pytest

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd._lib import IcsfError, check, lib, ptr
from icsfoam_amd.mesh import prepare_case
from icsfoam_amd.solver import hbCase

from helpers import bump_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 70])
def test_history_batches(n):
    print(f"[history {n}]", flush=True)
    c = bump_small(16, 8)
    a, b = dbnsCase.from_case(c), dbnsCase.from_case(c)
    h = a.pseudo_steps(n)
    one = np.concatenate([b.pseudo_steps(1) for _ in range(n)])
    np.testing.assert_array_equal(h, one)


@pytest.mark.parametrize("max_iter", [1, 2])
def test_hb_history_batches(max_iter):
    print(f"[hb history {max_iter}]", flush=True)
    insts, D, _ = cases.case_hb(n=(6, 4, 3), n_harmonics=1)
    insts = [dataclasses.replace(prepare_case(c, permute_seed=1), fvSolution=cases.solution_dict(
        co=20.0, nDirections=4, maxIter=max_iter, relTol=1e-6)) for c in insts]
    a, b = hbCase.from_cases(insts, D), hbCase.from_cases(insts, D)
    h = a.pseudo_steps(35)
    one = np.concatenate([b.pseudo_steps(1) for _ in range(35)])
    np.testing.assert_array_equal(h, one)
    F = a.fields(1)
    np.testing.assert_array_equal(F["W"][0], F["rho"])


def test_field_subsets():
    c = bump_small(20, 7)
    g = dbnsCase.from_case(c)
    g.pseudo_steps(2)
    full = g.fields()
    n = g.nCells
    np.testing.assert_array_equal(full["W"][0], full["rho"])
    np.testing.assert_allclose(full["W"][2:].T, full["rho"][:, None] * full["U"], rtol=1e-15)
    for mask in range(1, 32):
        out = [np.empty(n), np.empty((n, 3)), np.empty(n), np.empty(n), np.empty((5, n))]
        arg = [ptr(x) if mask >> i & 1 else None for i, x in enumerate(out)]
        check(lib().icsf_get_fields(g._h, *arg))
        for i, k in enumerate(("rho", "U", "T", "p", "W")):
            if mask >> i & 1:
                np.testing.assert_array_equal(out[i], full[k])


@pytest.mark.parametrize("nx,ny", [(102, 100), (128, 80), (128, 81), (160, 81)])
def test_field_subsets_on_both_sides_of_the_gather(nx, ny):
    """Cell counts around 10 240, above which the device gathers rho, p, U."""
    print(f"[fields {nx} x {ny}]", flush=True)
    g = dbnsCase.from_case(bump_small(nx, ny))
    g.pseudo_steps(1)
    n = g.nCells
    full = g.fields()
    np.testing.assert_array_equal(full["W"][0], full["rho"])
    np.testing.assert_allclose(full["W"][2:].T, full["rho"][:, None] * full["U"], rtol=1e-15)
    np.testing.assert_allclose(full["p"], cases.R_GAS * full["rho"] * full["T"], rtol=1e-14)
    for mask in (1, 2, 8, 11, 18, 25):
        out = [np.empty(n), np.empty((n, 3)), np.empty(n), np.empty(n), np.empty((5, n))]
        check(lib().icsf_get_fields(g._h, *[ptr(x) if mask >> i & 1 else None for i, x in enumerate(out)]))
        for i, k in enumerate(("rho", "U", "T", "p", "W")):
            if mask >> i & 1:
                np.testing.assert_array_equal(out[i], full[k])


def _fail_step(case=None, hb=None, step=0):
    """The next pseudo_steps fails at this step; a test entry beside the
    interface."""
    f = lib().icsf_test_fail_step
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    check(f(case, hb, step))


def _check_kept(kept, step, want):
    """Residual array left by a call that failed at `step`: the steps before
    it as asked for alone, those after it untouched."""
    np.testing.assert_array_equal(kept[:step], want)
    assert np.isnan(kept[step:]).all()


@pytest.mark.parametrize("step", [0, 1, 5, 32, 33, 40])
def test_failed_step_keeps_the_history_before_it(step):
    print(f"[history, step {step} fails]", flush=True)
    c = bump_small(16, 8)
    a, b = dbnsCase.from_case(c), dbnsCase.from_case(c)
    h = np.full((45, 10), np.nan)
    _fail_step(case=a._h, step=step)
    with pytest.raises(IcsfError):
        check(lib().icsf_pseudo_steps(a._h, 45, ptr(h), None))
    _check_kept(h, step, b.pseudo_steps(step))
    np.testing.assert_array_equal(a.pseudo_steps(3), b.pseudo_steps(3))  # and goes on from there


@pytest.mark.parametrize("max_iter", [1, 2])
def test_failed_hb_step_keeps_the_history_before_it(max_iter):
    print(f"[hb history, a step fails, {max_iter}]", flush=True)
    insts, D, _ = cases.case_hb(n=(6, 4, 3), n_harmonics=1)
    insts = [dataclasses.replace(prepare_case(c, permute_seed=1), fvSolution=cases.solution_dict(
        co=20.0, nDirections=4, maxIter=max_iter, relTol=1e-6)) for c in insts]
    a, b = hbCase.from_cases(insts, D), hbCase.from_cases(insts, D)
    h = np.full((10, 3, 10), np.nan)
    _fail_step(hb=a._h, step=7)
    with pytest.raises(IcsfError):
        check(lib().icsf_hb_pseudo_steps(a._h, 10, ptr(h)))
    _check_kept(h, 7, b.pseudo_steps(7))
    np.testing.assert_array_equal(a.pseudo_steps(2), b.pseudo_steps(2))


@pytest.mark.parametrize("n", [(6, 4, 3), (24, 22, 20)])
def test_hb_reads_between_steps(n):
    """Field read-backs gather in the system's work vector: every instance's
    own fields, and the steps that follow as without them."""
    print(f"[hb reads {n}]", flush=True)
    insts, D, _ = cases.case_hb(n=n, n_harmonics=1)
    insts = [prepare_case(c, permute_seed=1) for c in insts]
    a, b = hbCase.from_cases(insts, D), hbCase.from_cases(insts, D)
    h = []
    for _ in range(4):
        for J in (2, 0, 1):
            F = a.fields(J)
            np.testing.assert_array_equal(F["W"][0], F["rho"])
            np.testing.assert_allclose(F["W"][2:].T, F["rho"][:, None] * F["U"], rtol=1e-15)
            np.testing.assert_allclose(F["p"], cases.R_GAS * F["rho"] * F["T"], rtol=1e-14)
        h.append(a.pseudo_steps(1))
    np.testing.assert_array_equal(np.concatenate(h), b.pseudo_steps(4))
