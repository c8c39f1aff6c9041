"""LU-SGS of numberings with many dependency levels (one dataflow launch)
against the sequential sweep, bit for bit: RCM and file order, chunks of one
row and of a wavefront, level counts on both sides of where the launch per
level is left (24), generator and block storage, FP32 blocks with FP64 and with
FP32 vectors, and repeated applications (the values of one must not serve the
next).  And what calls do when a sweep gives up."""
import ctypes
import dataclasses

import numpy as np
import pytest

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd._lib import ERR_HIP, ERR_NONFINITE, IcsfError, check, lib
from icsfoam_amd.mesh import prepare_case
from oracle.oracle import OracleCase

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _case(n, order, **sol):
    c = cases.case_box(n=n, jitter=0.1, flux="ROE", mu=1.8e-5)
    if order == "rcm":
        c = prepare_case(c, permute_seed=5, colour_major=False)
    return dataclasses.replace(c, fvSolution=cases.solution_dict(**sol))


@pytest.mark.parametrize("storage", ["generators", "blocks"])
@pytest.mark.parametrize("n,order", [((3, 1, 1), "file"), ((11, 1, 1), "file"), ((12, 1, 1), "file"),
                                     ((70, 1, 1), "file"), ((9, 8, 7), "rcm"), ((16, 16, 9), "file"), ((33, 20, 17), "rcm")])
def test_many_level_sweep_is_the_sequential_one(n, order, storage):
    print(f"[sweep {n} {order} {storage}]", flush=True)
    c = _case(n, order, jacobianStorage=storage)
    g, o = dbnsCase.from_case(c), OracleCase(c)
    # 24 levels in all and more take the dataflow launch
    assert (g.mesh.nFwdLevels + g.mesh.nBwdLevels >= 24) == (n not in ((3, 1, 1), (11, 1, 1)))
    g.residual()
    o.residual()
    g.createJacobian()
    o.createJacobian()
    rng = np.random.default_rng(1)
    for _ in range(3):
        x = rng.standard_normal((5, g.nCells))
        np.testing.assert_array_equal(g.precondition(x), o.precondition(x))


MIXED = dict(solver="FGMRES", nDirections=1, precision="mixed")


@pytest.mark.parametrize("n,order", [((12, 1, 1), "file"), ((14, 9, 8), "rcm"), ((16, 16, 9), "file")])
def test_fp32_blocks_fp64_vectors(n, order):
    """The oracle given the FP32 blocks does the same FP64 operations."""
    print(f"[sweep fp32 blocks {n} {order}]", flush=True)
    c = _case(n, order, jacobianStorage="blocks", **MIXED)
    g, o = dbnsCase.from_case(c), OracleCase(c)
    g.residual()
    g.createJacobian()
    J = g.jacobian()
    g.set_jacobian(*J)  # rD from the rounded diagonal, as the oracle's
    o.set_matrix(*J)
    x = np.random.default_rng(1).standard_normal((5, g.nCells))
    np.testing.assert_array_equal(g.precondition(x), o.precondition(x))


def _sweep32(m, d, u, l, r):
    """Sequential LU-SGS in FP32, operations and order of a row as the
    kernels': r -> f (lower neighbours upwards) -> result (upper neighbours
    downwards)."""
    nC, own, nei = m.n_cells, m.owner[:m.n_internal], m.neighbour
    rD = np.full(nC, 1e15)
    for q in range(5):
        rD = 1.0 / np.maximum(1.0 / rD, np.abs(d[:, q, q]))
    rD, u, l, r = (np.asarray(a, np.float32) for a in (rD, u, l, r))
    lower, upper = [[] for _ in range(nC)], [[] for _ in range(nC)]
    for f in range(m.n_internal):
        lower[nei[f]].append((own[f], l[f]))
        upper[own[f]].append((nei[f], u[f]))

    def sub(acc, B, x):
        acc = (acc - B[:, 0] * x[0]) - B[:, 1] * x[1]
        return acc - ((B[:, 2] * x[2] + B[:, 3] * x[3]) + B[:, 4] * x[4])

    f, o = np.empty((nC, 5), np.float32), np.empty((nC, 5), np.float32)
    for c in range(nC):
        f[c] = r[:, c]
        for p, B in sorted(lower[c], key=lambda t: t[0]):
            f[c] = sub(f[c], B, rD[p] * f[p])
    for c in range(nC - 1, -1, -1):
        a = f[c]
        for q, B in sorted(upper[c], key=lambda t: -t[0]):
            a = sub(a, B, o[q])
        o[c] = rD[c] * a
    return o.T


@pytest.mark.parametrize("storage", ["generators", "blocks"])
@pytest.mark.parametrize("n,order", [((12, 1, 1), "file"), ((14, 9, 8), "rcm"), ((16, 16, 9), "file")])
def test_fp32_vectors(n, order, storage):
    """One flexible direction preconditioned by the FP32 sweep alone: the
    increment is that sweep of b / |b|, in FP32, times a scalar.  Its blocks
    are the case's; its scalar diagonal is that of the FP64 diagonal."""
    print(f"[sweep fp32 {n} {order} {storage}]", flush=True)
    c = _case(n, order, jacobianStorage=storage, innerDirections=0, **MIXED)
    g, o = dbnsCase.from_case(c), OracleCase(_case(n, order))
    b, _ = g.residual()
    o.residual()
    g.createJacobian()
    dW = g.solveForIncr(b=b)[0]
    _, u, l = g.jacobian()
    z = _sweep32(c.mesh, o.createJacobian()[0], u, l, b / np.sqrt((b * b).sum())).astype(np.float64)
    k = np.unravel_index(np.abs(z).argmax(), z.shape)
    y = dW[k] / z[k]
    # y z rounds once, as does y formed here: two units in the last place
    np.testing.assert_allclose(dW, y * z, rtol=2.0 ** -51, atol=0)


@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_many_level_pseudo_steps(form):
    print(f"[sweep steps {form}]", flush=True)
    kw = dict() if form == "fp64" else dict(solver="FGMRES", nDirections=1, precision="mixed", innerDirections=30)
    c = _case((14, 9, 8), "rcm", **kw)
    g = dbnsCase.from_case(c)
    e = dbnsCase.from_case(dataclasses.replace(c, fvSolution=cases.solution_dict(graphCapture=False, **kw)))
    h = g.pseudo_steps(5)
    np.testing.assert_array_equal(h, e.pseudo_steps(5))  # replayed = eager
    np.testing.assert_array_equal(g.fields()["W"], e.fields()["W"])
    o = OracleCase(_case((14, 9, 8), "rcm"))
    ho = o.pseudo_steps(5)
    # each conserved row and initial residual on its own scale; the final
    # residuals, differences b - A dW down to 1e-10 of the initial ones, carry
    # the initial ones' rounding
    tol = 1e-8 if form == "fp64" else 1e-3
    for a, b in zip(g.fields()["W"], o.fields()["W"]):
        assert rel_err(a, b) < tol
    for a, b in zip(h.T[:5], ho.T[:5]):
        assert rel_err(a, b) < tol
    assert abs(h - ho).max() < tol * abs(ho).max()


def _sweep_limit(g, polls):
    """Polls after which one wait of the sweep gives up (negative: the
    default); a test entry beside the interface."""
    f = lib().icsf_test_sweep_limit
    f.argtypes = [ctypes.c_void_p, ctypes.c_int]
    check(f(g._h, polls))


def test_wait_limit_is_per_wait():
    """A chain of single-cell levels: every wavefront draws 157 of the 40 000
    chunks and waits each time for at most the 256 chunks in flight (some 500
    polls; the whole sweep some 80 000).  A limit of 20 000 polls per wait
    must not end it."""
    print("[sweep limit]", flush=True)
    c = _case((20000, 1, 1), "file")
    g, o = dbnsCase.from_case(c), OracleCase(c)
    assert g.mesh.nFwdLevels == g.nCells
    for q in (g, o):
        q.residual()
        q.createJacobian()
    _sweep_limit(g, 20000)
    x = np.random.default_rng(1).standard_normal((5, g.nCells))
    np.testing.assert_array_equal(g.precondition(x), o.precondition(x))


def _gives_up(call):
    with pytest.raises(IcsfError, match="sweep") as e:
        call()
    assert e.value.code == ERR_HIP


def test_sweep_that_gives_up_is_reported():
    """A sweep whose waits may not wait (limit 0) gives up: every call that
    ran it reports that, none hands its failure to a later call, and with the
    limit back the same calls give the same bits as before."""
    print("[sweep gives up]", flush=True)
    c = _case((16, 16, 9), "file")
    g = dbnsCase.from_case(c)
    g.residual()
    g.createJacobian()
    x = np.random.default_rng(1).standard_normal((5, g.nCells))
    p, (dW, res, _) = g.precondition(x), g.solveForIncr()
    _sweep_limit(g, 0)
    _gives_up(g.solveForIncr)
    _sweep_limit(g, -1)
    np.testing.assert_array_equal(g.precondition(x), p)
    _sweep_limit(g, 0)
    _gives_up(lambda: g.precondition(x))
    _sweep_limit(g, -1)
    d, r, _ = g.solveForIncr()
    np.testing.assert_array_equal(d, dW)
    np.testing.assert_array_equal(r, res)
    _sweep_limit(g, 0)
    _gives_up(lambda: g.pseudo_steps(4))  # the last ones replayed
    _gives_up(lambda: g.pseudo_time_loop(2))


def test_sweep_that_gives_up_is_the_cause_reported():
    """With an inflow whose |U|^2 overflows the state turns non-finite too:
    the sweep is the cause reported, and without it the state is."""
    print("[sweep gives up, non-finite]", flush=True)
    c = _case((16, 16, 9), "file")
    i = [p.name for p in c.mesh.patches].index("inlet")
    U = np.zeros((c.mesh.patches[i].size, 3))
    U[:, 0] = 1e200
    bcs = list(c.bcs)
    bcs[i] = dataclasses.replace(bcs[i], U_val=U)
    g = dbnsCase.from_case(dataclasses.replace(c, bcs=bcs))
    _sweep_limit(g, 0)
    _gives_up(lambda: g.pseudo_steps(2))
    g = dbnsCase.from_case(dataclasses.replace(c, bcs=bcs))
    with pytest.raises(IcsfError) as e:
        g.pseudo_steps(2)
    assert e.value.code == ERR_NONFINITE
