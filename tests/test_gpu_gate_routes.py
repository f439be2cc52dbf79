"""The learned limiter's routes on one simulation, one after the other: a whole stage, a stage in two calls,
a stage with capture and a stage with the judge, bit for bit what a simulation that is always judged holds."""
import numpy as np
import pytest

from dgswemv2_amd import RKDG_FP32_BULK, RKDG_FP64_FAST, RKDG_FP64_PLAIN, Simulation
from dgswemv2_amd import indicator as IND
from dgswemv2_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,precision,stages", [(1, RKDG_FP64_PLAIN, 16), (1, RKDG_FP64_FAST, 16), (1, RKDG_FP32_BULK, 16),
                                                (2, RKDG_FP64_PLAIN, 8), (2, RKDG_FP32_BULK, 8)])
def test_alternating_routes_equal_always_judged(p, precision, stages):
    mesh, prm = W.dambreak(scale=0.1, p=p)
    net = IND.init_weights(11)
    a, b = Simulation(mesh, prm, precision), Simulation(mesh, prm, precision)
    for s in (a, b):
        s.step(4)
    # a threshold that opens some 30 % of the elements the limiter may act on
    t = Simulation(mesh, prm, precision)
    t.set_indicator(net, threshold=-3.0e38)
    t.capture(True)
    t.step(5)
    c = t.get_capture(logits=True)
    t.close()
    thr = float(np.quantile(c["logit"][c["may_act"] != 0], 0.7))
    a.set_indicator(net, threshold=thr, judge=True)
    b.set_indicator(net, threshold=thr)

    def whole():
        b.stage()

    def in_two():
        b.stage_begin()
        b.stage_finish()

    def captured():
        b.capture(True)
        b.stage()
        b.capture(False)

    def judged():
        b.set_indicator(net, threshold=thr, judge=True)
        b.stage()
        b.set_indicator(net, threshold=thr)

    routes = (whole, in_two, whole, captured, in_two, judged, whole, in_two)
    limited = 0
    for k in range(stages):
        print("[gpu-gate-routes] p", p, "precision", precision, "stage", k, routes[k % 8].__name__, flush=True)
        a.stage()
        routes[k % 8]()
        sa, sb = a.state(), b.state()
        for f in ("q", "wet", "limited", "troubled"):
            assert np.array_equal(sa[f], sb[f]), (k, routes[k % 8].__name__, f)
        limited += int(sa["limited"].any(axis=0).sum())
    st = a.indicator_stats()
    assert 0 < st["flagged"] < st["candidates"] and limited > 0, (st, limited)
    a.close(), b.close()
