"""States of 26 to 70 MB through set_state and state: three, five and eight readers, the chunks of a write before
and after a reading, and ensembles whose instances need more readers or a flag copy of their own."""
import numpy as np
import pytest

from dgswemv2_amd import (BC_LAND, RKDG_FP32_BULK, RKDG_FP64_FAST, RKDG_FP64_PLAIN, Batch, Simulation, make_params,
                          quad_mesh)

pytestmark = pytest.mark.gpu


def _case(m, p, limiting=False):
    mesh = quad_mesh(0.0, 0.0, m, m, m, m, bc=(BC_LAND,) * 4, bathy="constant", b0=3.0, jitter=0.1, seed=2)
    return mesh, make_params(p=p, nstages=2, order=2, dt=1e-6, g=9.81, wetting_drying=limiting, h_o=0.01,
                             slope_limiting=limiting, sl_M=1e30)


def _state(ne, p, seed, single):
    q = np.random.default_rng(seed).uniform(-1.0, 1.0, (3, (p + 1) * (p + 2) // 2, ne))
    return q.astype(np.float32).astype(np.float64) if single else q


@pytest.mark.parametrize("m,p,precision", [(300, 2, RKDG_FP64_FAST), (400, 2, RKDG_FP64_FAST), (490, 2, RKDG_FP64_FAST),
                                           (490, 2, RKDG_FP32_BULK), (700, 1, RKDG_FP64_PLAIN)])
def test_large_states_come_back(m, p, precision):
    print("[gpu-transfer] m", m, "p", p, "precision", precision, flush=True)
    mesh, prm = _case(m, p)
    s = Simulation(mesh, prm, precision)
    for seed in (1, 2, 3):  # the first is written before anything was read
        q = _state(mesh.n_elements, p, seed, precision == RKDG_FP32_BULK)
        s.set_state(q)
        assert np.array_equal(s.state()["q"], q), seed
    # written twice with a reading's buffers still in use by the first
    a, b = (_state(mesh.n_elements, p, seed, precision == RKDG_FP32_BULK) for seed in (4, 5))
    s.set_state(a)
    s.set_state(b)
    assert np.array_equal(s.state()["q"], b)
    s.close()


def test_ensemble_instances_of_growing_size_come_back():
    cases = [_case(m, 2) for m in (60, 300, 490)]
    b = Batch([c[0] for c in cases], [c[1] for c in cases], RKDG_FP64_FAST)
    for round_ in range(2):
        qs = [_state(c[0].n_elements, 2, 10 * round_ + i, False) for i, c in enumerate(cases)]
        for i, q in enumerate(qs):
            b.set_state(i, q)
        for i, q in enumerate(qs):
            print("[gpu-transfer] ensemble instance", i, flush=True)
            assert np.array_equal(b.state(i)["q"], q), i
    b.close()


def test_flags_of_a_large_instance_equal_its_single_run():
    # 5 flag bytes an element: above 52,428 elements they do not fit the staged copy
    cases = [_case(m, 1, limiting=True) for m in (40, 170)]
    assert cases[1][0].n_elements > 52428
    b = Batch([c[0] for c in cases], [c[1] for c in cases], RKDG_FP64_PLAIN)
    ref = []
    for i, (mesh, prm) in enumerate(cases):
        ne = mesh.n_elements
        rng = np.random.default_rng(7 + i)
        q = np.zeros((3, 3, ne))
        q[0, 0] = 1.5 * (rng.random(ne) < 0.01) * rng.choice([-1, 1], ne)
        q[1, 0] = 1e-3
        wet = np.ones(ne, np.uint8)
        s = Simulation(mesh, prm, RKDG_FP64_PLAIN)
        s.set_state(q, wet)
        s.step(2)
        ref.append(s.state())
        s.close()
        b.set_state(i, q, wet)
    b.step(2)
    for i, r in enumerate(ref):
        got = b.state(i)
        print("[gpu-transfer] flags of instance", i, "limited", r["limited"].mean(), "troubled", r["troubled"].mean(), flush=True)
        assert 0.0 < r["limited"].mean() < 1.0 and 0.0 < r["troubled"].mean() < 1.0
        for f in ("q", "wet", "limited", "troubled"):
            assert np.array_equal(got[f], r[f]), (i, f)
    b.close()
