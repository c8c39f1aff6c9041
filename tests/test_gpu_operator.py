"""Fused Arnoldi operator (SpMV and LU-SGS sweeps of a two-colour numbering)
against the separate kernels: row counts below, at and above a wavefront and
a workgroup, a two-colour numbering whose levels are no cell ranges, and
matrices with a frame-zone term and with cyclic interfaces.

Only the order of a row's sums differs, so GMRES increments agree to 1e-12
in FP64 and 1e-4 with the FP32 inner solve (the bounds of
test_fused_spmv_lusgs_matches_unfused)."""
import dataclasses

import numpy as np
import pytest

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd.mesh import colour_cells, prepare_case, renumber_mesh

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _interleaved(case):
    """Colour-1 cells right after their last colour-0 neighbour: two sweep
    levels, neither of them a range of cells."""
    m = case.mesh
    col, n = colour_cells(m)
    assert n == 2
    nbr = [[] for _ in range(m.n_cells)]
    for o, p in zip(m.owner[:m.n_internal], m.neighbour):
        nbr[o].append(p)
        nbr[p].append(o)
    left = {c: len(nbr[c]) for c in range(m.n_cells) if col[c] == 1}
    order = []
    for c in np.flatnonzero(col == 0):
        order.append(c)
        for p in nbr[c]:
            left[p] -= 1
            if left[p] == 0:
                order.append(p)
    return cases.permute_case(case, np.array(order, np.int32), renumber_mesh)


def _check(c, **kw):
    gs = []
    for fused in (True, False):
        g = dbnsCase.from_case(dataclasses.replace(c, fvSolution=cases.solution_dict(fusedSweeps=fused, **kw)))
        assert g.mesh.nFwdLevels == 2 and g.mesh.nBwdLevels == 2
        g.residual()
        g.createJacobian()
        gs.append(g.solveForIncr())
    tol = 1e-4 if kw.get("precision") == "mixed" else 1e-12
    assert rel_err(gs[0][0], gs[1][0]) < tol
    assert rel_err(gs[0][1], gs[1][1]) < tol


MIXED = dict(solver="FGMRES", nDirections=2, precision="mixed", innerDirections=12)


@pytest.mark.parametrize("kw", [dict(nDirections=12), MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", [(2, 1, 1), (5, 5, 5), (8, 4, 4), (17, 16, 15), (64, 47, 46)])
def test_fused_operator_row_counts(n, kw):
    print(f"[operator {n} {sorted(kw)}]", flush=True)
    if n == (2, 1, 1):
        kw = dict(kw, **({"innerDirections": 2} if "innerDirections" in kw else {"nDirections": 2}))
    _check(prepare_case(cases.case_box(n=n, jitter=0.1, flux="ROE", mu=1.8e-5), permute_seed=2), **kw)


@pytest.mark.parametrize("kw", [dict(nDirections=12), MIXED], ids=["fp64", "mixed"])
def test_fused_operator_levels_not_ranges(kw):
    print("[operator interleaved]", flush=True)
    _check(_interleaved(cases.case_box(n=(7, 6, 5), jitter=0.1, flux="ROE", mu=1.8e-5)), **kw)


@pytest.mark.parametrize("storage", ["generators", "blocks"])
@pytest.mark.parametrize("kw", [dict(nDirections=12), MIXED], ids=["fp64", "mixed"])
def test_fused_operator_rotating_cyclic_sector(kw, storage):
    print(f"[operator sector {storage}]", flush=True)
    c = prepare_case(cases.case_sector(nt=8, nr=6, nz=5), permute_seed=2)
    c.mrf = cases.MRFZone(np.ones(c.mesh.n_cells, bool), np.zeros(3), np.array([0.0, 0.0, 1.0]), 120.0,
                          list(range(len(c.mesh.patches))))
    _check(c, jacobianStorage=storage, **kw)
