"""An open boundary whose given surface lies below the bed: the FP64 forms against the oracle.

Where a tide falls below the bed of a wet boundary element the exterior depth is negative.  Its wave speed
is the square root of a negative number, which the maximum over the two sides passes over (std::max with the
interior's speed first); its velocity is the discharge over the negative depth.  Every flux is finite.

Tolerance: one stage of the fast form against the oracle, as for the other tidal runs (1e-12 of each
variable's norm); the plain form, whose cosine may differ by a unit, to 1e-14.
"""
import numpy as np
import pytest

from conftest import relerr
from dgswemv2_amd import BC_LAND, BC_TIDE, RKDG_FP64_FAST, RKDG_FP64_PLAIN, Simulation, make_params, quad_mesh
from oracle.oracle_py import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,tol", [(RKDG_FP64_PLAIN, 1e-14), (RKDG_FP64_FAST, 1e-12)])
@pytest.mark.parametrize("p", [1, 2, 3])
def test_surface_given_below_the_bed(p, form, tol):
    mesh = quad_mesh(0.0, 0.0, 700.0, 500.0, 7, 5, bc=(BC_LAND, BC_LAND, BC_LAND, BC_TIDE), bathy="constant", b0=1.0, jitter=0.1, seed=4,
                     frequency=1e-4, amplitude=1.3, phase=180.0)
    prm = make_params(p=p, nstages=2, order=2, dt=0.5, g=9.81)
    g, o = Simulation(mesh, prm, form), OracleSim(mesh, prm)
    q = g.state()["q"]
    rng = np.random.default_rng(5)
    q[0, 0] = 0.05 * rng.uniform(-1, 1, mesh.n_elements)
    q[1:, :3] = 0.1 * rng.uniform(-1, 1, (2, 3, mesh.n_elements))
    g.set_state(q), o.set_state(q, np.ones(mesh.n_elements, np.uint8))
    print("[gpu-open]", p, form, flush=True)
    g.stage(), o.stage()
    a, b = g.state()["q"], o.state()["q"]
    assert np.isfinite(b).all() and np.isfinite(a).all()
    assert max(relerr(a, b)) <= tol
    g.close(), o.close()
