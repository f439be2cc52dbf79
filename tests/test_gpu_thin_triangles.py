"""Bottom friction of the fast forms on thin, turned triangles.

The friction integral carries |det J|.  On a triangle with a small angle that is not aligned with the
axes, a determinant formed from rounded matrix entries is a difference of nearly equal products; the fast
forms have to use the one the mesh gives.  A uniform flow over a flat bed changes by friction alone where
no face lies on the boundary: after one forward-Euler step q = q0 (1 - dt cf |u| / h), with cf one: Chezy's,
Manning's g n^2 / h^(1/3), or its floor.

Tolerance: a friction term of 0.3 q0 is the product of a root, a reciprocal (each within one unit of
rounding), about twelve rounded factors and a quadrature sum: 32 roundings of 0.3 q0, and two of q0 for the
update.  Fluxes of a uniform state cancel to rounding, times dt |u| / height = 0.05 at most.
"""
import numpy as np
import pytest

from dgswemv2_amd import (BC_LAND, FRICTION_CHEZY, FRICTION_MANNING, RKDG_FP32_BULK, RKDG_FP64_FAST, RKDG_FP64_PLAIN, Simulation,
                          make_params, quad_mesh)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [RKDG_FP64_PLAIN, RKDG_FP64_FAST, RKDG_FP32_BULK])
@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("law", ["chezy", "manning", "manning floor"])
@pytest.mark.parametrize("aspect", [1.0, 20.0, 200.0])
def test_friction_on_thin_triangles(aspect, law, p, form):
    mesh = quad_mesh(0.0, 0.0, 12.0, 10.0, 12, 10, bc=(BC_LAND,) * 4, bathy="constant", b0=1.0, jitter=0.2, seed=3,
                     manning_n=1.0 / np.sqrt(9.81) if law == "manning" else 0.1)
    x, y, turn = 10.0 * aspect * mesh.node_xyz[:, 0], 10.0 * mesh.node_xyz[:, 1], np.deg2rad(37.0)
    mesh.node_xyz[:, 0], mesh.node_xyz[:, 1] = np.cos(turn) * x - np.sin(turn) * y, np.sin(turn) * x + np.cos(turn) * y
    dt, u, v = 3.0, 0.08, -0.06
    prm = make_params(p=p, nstages=1, order=1, dt=dt, g=9.81, friction=FRICTION_CHEZY if law == "chezy" else FRICTION_MANNING,
                      friction_cf=0.0 if law == "manning" else 1.0)
    s = Simulation(mesh, prm, form)
    q = np.zeros((3, (p + 1) * (p + 2) // 2, mesh.n_elements))
    q[1, 0], q[2, 0] = (np.float32(z).astype(np.float64) for z in (u, v))
    q0 = q[:, 0, 0].copy()
    s.set_state(q)
    print("[gpu-thin]", aspect, law, p, form, flush=True)
    s.stage()
    got = s.state()["q"]
    s.close()
    # elements without a boundary face: each of their edges belongs to two
    e = np.sort(np.stack([mesh.elt_nodes.reshape(-1, 3)[:, [a, b]] for a, b in ((0, 1), (1, 2), (2, 0))], 1), 2)
    _, where, count = np.unique(e.reshape(-1, 2), axis=0, return_inverse=True, return_counts=True)
    inner = (count[where.reshape(-1)].reshape(-1, 3) == 2).all(1)
    assert inner.sum() > 100
    unit = 2.0**-24 if form == RKDG_FP32_BULK else 2.0**-53
    speed = np.hypot(*q0[1:])
    tol = (32 * 0.3 + 2 + 8 * 0.05) * unit * speed
    for k in (1, 2):
        want = q0[k] * (1.0 - dt * speed)
        assert np.max(np.abs(got[k, 0, inner] - want)) <= tol, (k, np.max(np.abs(got[k, 0, inner] - want)) / tol)
