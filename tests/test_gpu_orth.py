"""Gram-Schmidt step of the device GMRES against the oracle's modified
Gram-Schmidt, over the edges of its chunks: one and two directions, one more
than a chunk of 8, 16 and 32 basis vectors, the largest cycle; cells no
multiple of a wavefront, and cell counts on both sides of where the update
sums the projection partials itself and changes its workgroup size.

Both forms span the oracle's Krylov space, so the increments agree to the
rounding of the orthogonalisation: modified Gram-Schmidt (one pass, inverse
compact WY) 1e-10 and classical 1e-8 as elsewhere for these solves."""
import dataclasses

import pytest

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd.mesh import prepare_case
from oracle.oracle import OracleCase

from helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("orth", ["MGS", "CGS"])
@pytest.mark.parametrize("n,dirs", [((11, 9, 7), d) for d in (1, 2, 9, 17, 33, 64)] +
                         [((28, 23, 20), 5), ((33, 23, 17), 5), ((28, 25, 24), 18)])
def test_gram_schmidt_chunk_edges(n, dirs, orth):
    c = prepare_case(cases.case_box(n=n, jitter=0.1, flux="ROE", mu=1.8e-5), permute_seed=4)
    print(f"[orth {n} {orth} {dirs}]", flush=True)
    c = dataclasses.replace(c, fvSolution=cases.solution_dict(nDirections=dirs, orthogonalisation=orth))
    g, o = dbnsCase.from_case(c), OracleCase(c)
    g.residual()
    bo, _ = o.residual()
    g.createJacobian()
    o.createJacobian()
    dWg, rg, _ = g.solveForIncr()
    dWo, ro, _ = o.solveForIncr(g.fields()["W"], bo)
    tol = 1e-10 if orth == "MGS" else 1e-8
    assert rel_err(dWg, dWo) < tol
    # the last residuals, relative to the first ones (64 directions reach
    # rounding level)
    assert abs(rg - ro).max() < tol * abs(ro).max()
