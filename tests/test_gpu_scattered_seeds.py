"""Trouble seeds scattered over the mesh, from none to nearly everywhere: the troubled flags, the limited flags
and the state after a stage equal the oracle's, alone and in an ensemble under each work-group size."""
import numpy as np
import pytest

from dgswemv2_amd import BC_LAND, RKDG_FP64_PLAIN, Batch, Simulation, make_params, quad_mesh
from oracle.oracle_py import OracleSim

pytestmark = pytest.mark.gpu


def _case(m, density):
    mesh = quad_mesh(0.0, 0.0, m, m, m, m, bc=(BC_LAND,) * 4, bathy="constant", b0=3.0, jitter=0.1, seed=2)
    prm = make_params(p=1, nstages=2, order=2, dt=1e-6, g=9.81, wetting_drying=True, h_o=0.01, slope_limiting=True, sl_M=1e30)
    o = OracleSim(mesh, prm)
    ne = mesh.n_elements
    rng = np.random.default_rng(int(1000 * density) + m)
    q = o.state()["q"]
    q[0, 0] += 1.5 * (rng.random(ne) < density) * rng.choice([-1, 1], ne)
    q[1, 0] = 1e-3
    wet = np.ones(ne, np.uint8)
    o.set_state(q, wet)
    o.step(1)
    ref = o.state()
    o.close()
    return mesh, prm, q, wet, ref


@pytest.mark.parametrize("density", [0.0, 0.002, 0.03, 0.2, 0.5, 0.9])
def test_scattered_seeds_match_oracle(density):
    cases = [_case(m, density) for m in (9, 40)]
    share = [r["troubled"].mean() for *_, r in cases]
    if density == 0.0:
        assert max(share) == 0.0
    elif density >= 0.03:
        assert share[1] > 0.2
    print("[gpu-scattered-seeds] density", density, "troubled", share, flush=True)
    for mesh, prm, q, wet, ref in cases:
        s = Simulation(mesh, prm, RKDG_FP64_PLAIN)
        s.set_state(q, wet)
        s.step(1)
        got = s.state()
        s.close()
        for f in ("q", "wet", "limited", "troubled"):
            assert np.array_equal(got[f], ref[f]), (mesh.n_elements, f)
    for block in (64, 128, 256):
        print("[gpu-scattered-seeds] ensemble, block", block, flush=True)
        b = Batch([c[0] for c in cases], [c[1] for c in cases], RKDG_FP64_PLAIN)
        b.set_schedule(block=block, groups_per_xcd=0, graph=0)
        for i, (_, _, q, wet, _) in enumerate(cases):
            b.set_state(i, q, wet)
        b.step(1)
        for i, (*_, ref) in enumerate(cases):
            got = b.state(i)
            for f in ("q", "wet", "limited", "troubled"):
                assert np.array_equal(got[f], ref[f]), (block, i, f)
        b.close()
