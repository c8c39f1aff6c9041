"""icsf_residual_device writes short face records and updates the state straight
from the caller's W: the residual is icsf_residual's bit for bit, the Jacobian
and pseudo-steps that follow it are those after icsf_residual, and W may be
the output array; every scheme, viscous and inviscid, second and first order,
cell counts at the edges of a wavefront."""
import numpy as np
import pytest
import torch

from icsfoam_amd import cases, dbnsCase
from icsfoam_amd._lib import check, lib
from icsfoam_amd.adjoint import residual_device
from icsfoam_amd.mesh import prepare_case

from helpers import ausm_inviscid, bump_small, hllc, roe

pytestmark = pytest.mark.gpu


def _cases():
    box = lambda n: prepare_case(cases.case_box(n=n, jitter=0.1 if min(n) > 1 else 0.0), permute_seed=1)  # noqa: E731
    return {
        "roe_visc": lambda: box((7, 6, 5)), "roe": lambda: roe(box((4, 4, 4)), mu=0.0),
        "ausm": lambda: ausm_inviscid(box((13, 5, 1))), "ausm_upwind": lambda: ausm_inviscid(box((11, 3, 2)), recon="upwind"),
        "hllc": lambda: hllc(box((5, 5, 5)), mu=0.0), "hllc_visc": lambda: hllc(box((43, 3, 1)), mu=1e-3),
        "bump": bump_small, "sector_visc": lambda: prepare_case(cases.case_sector(mu=1e-3), permute_seed=3),
    }


@pytest.mark.parametrize("which", sorted(_cases()))
def test_residual_device_equals_residual(which):
    print(f"[residual device {which}]", flush=True)
    c = _cases()[which]()
    g, h = dbnsCase.from_case(c), dbnsCase.from_case(c)
    W = torch.from_numpy(h.fields()["W"]).cuda() * (1 + 1e-3 * torch.rand(5, h.nCells, dtype=torch.float64).cuda())
    b = residual_device(g, W)
    h.set_state(W.cpu().numpy())
    bh, rdt = h.residual()
    np.testing.assert_array_equal(b.cpu().numpy(), bh)
    # the Jacobian of the same state, with the local time step
    g.createJacobian()
    h.createJacobian()
    for x, y in zip(g.jacobian(), h.jacobian()):
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(g.pseudo_steps(4), h.pseudo_steps(4))
    np.testing.assert_array_equal(g.fields()["W"], h.fields()["W"])
    # in place: W is the output
    g.set_state(W.cpu().numpy())
    X = W.clone()
    torch.cuda.synchronize()
    check(lib().icsf_residual_device(g._h, X.data_ptr(), X.data_ptr()))
    np.testing.assert_array_equal(X.cpu().numpy(), residual_device(h, W).cpu().numpy())
