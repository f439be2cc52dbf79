"""Wetting-drying ensembles with the limiter in the fast forms: every order, one work-group a tile and
persistent, each instance bit for bit its own single run.

The dam breaks have dry elements beyond the flood plain's edge, so that waves hold wet and dry lanes; the
instances differ in size, so that a wrong instance number shows.
"""
import numpy as np
import pytest

from dgswemv2_amd import RKDG_FP32_BULK, RKDG_FP64_FAST, Batch, Simulation, workloads as W

pytestmark = pytest.mark.gpu

SCHEDULES = [dict(block=128, groups_per_xcd=0, graph=0), dict(block=64, groups_per_xcd=-1, graph=0),
             dict(block=256, groups_per_xcd=-1, graph=1)]
STEPS = 8


@pytest.mark.parametrize("precision", [RKDG_FP64_FAST, RKDG_FP32_BULK])
@pytest.mark.parametrize("p", [1, 2, 3])
def test_wet_dry_ensemble_equals_single_runs(p, precision):
    cases = [W.dambreak(scale=scale, p=p) for scale in (0.04, 0.06, 0.05)]
    ref = []
    for mesh, prm in cases:
        s = Simulation(mesh, prm, precision)
        s.step(STEPS)
        ref.append(s.state())
        s.close()
    assert all(0 < (r["wet"] == 0).sum() < r["wet"].size and r["limited"].any() for r in ref)
    for sc in SCHEDULES:
        print("[gpu-batch-wet-dry] p", p, "precision", precision, sc, flush=True)
        b = Batch([c[0] for c in cases], [c[1] for c in cases], precision)
        b.set_schedule(**sc)
        b.step(STEPS)
        for i, r in enumerate(ref):
            got = b.state(i)
            for f in ("q", "wet", "limited", "troubled"):
                assert np.array_equal(got[f], r[f]), (sc, i, f)
        b.close()
