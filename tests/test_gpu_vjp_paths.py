"""The residual VJP with and without the geometry adjoint takes different
kernels for the Gauss face values (a face pass, or the cell pass itself): gW
must be the same bits, for every scheme, limiter state and cell counts at the
edges of a wavefront and of a workgroup."""
import numpy as np
import pytest

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd.mesh import prepare_case

from helpers import ausm_inviscid, hllc, roe

pytestmark = pytest.mark.gpu

SCHEMES = {"ausm": ausm_inviscid, "roe": lambda c, **k: roe(c, mu=0.0, **k), "hllc": lambda c, **k: hllc(c, mu=0.0, **k)}


@pytest.mark.parametrize("recon", ["linearUpwind limitedGrad", "upwind"])
@pytest.mark.parametrize("scheme", sorted(SCHEMES))
@pytest.mark.parametrize("n", [(2, 1, 1), (7, 3, 3), (4, 4, 4), (13, 5, 1), (16, 8, 1), (43, 3, 1), (12, 11, 10)])
def test_gW_same_bits_with_and_without_geometry(n, scheme, recon):
    print(f"[vjp paths {n} {scheme} {recon}]", flush=True)
    c = prepare_case(SCHEMES[scheme](cases.case_box(n=n, jitter=0.1 if min(n) > 1 else 0.0), recon=recon),
                     permute_seed=1)
    g = dbnsCase.from_case(c)
    W = g.fields()["W"]
    rng = np.random.default_rng(3)
    W = W * (1 + 1e-3 * rng.standard_normal(W.shape))
    v = rng.standard_normal(W.shape)
    a = g.residual_vjp(v, W, geometry=True)[0]
    b = g.residual_vjp(v, W, geometry=False)[0]
    assert np.isfinite(a).all() and np.abs(a).max() > 0
    np.testing.assert_array_equal(a, b)
