"""The indicator network where its sums overflow: a hidden unit without a number counts as zero."""
import numpy as np
import pytest

from dgswemv2_amd import indicator as IND
from dgswemv2_amd.indicator import MlpTrainer
from oracle import mlp as O

pytestmark = pytest.mark.gpu

FLT_MAX = float(np.finfo(np.float32).max)


def _reference(prm, X):
    h = O.bf16(X)
    with np.errstate(invalid="ignore", over="ignore"):
        for w, b in (("w1", "b1"), ("w2", "b2"), ("w3", "b3")):
            z = O.bf16(prm[w]) @ h + prm[b][:, None]
            z = np.where(np.abs(z) > FLT_MAX, np.sign(z) * np.inf, z)  # the sums are 32-bit floats
            h = np.where(z > 0, z, 0.0)
            if w != "w3":
                h = np.where(np.isfinite(h), O.bf16(h), h)
        return prm["w4"] @ h + prm["b4"]


@pytest.mark.parametrize("n", [5, 333])
def test_forward_counts_units_without_a_number_as_zero(n):
    # every product of such a sample's first layer is past the largest float, with one sign in a unit: units of
    # +inf and -inf, whose weighted sums in the second layer are no numbers
    print("network forward, overflowing features, n", n, flush=True)
    rng = np.random.default_rng(3)
    prm = O.unflatten(IND.init_weights(7) + 0.1 * rng.standard_normal(O.NPARAM))
    prm["w1"] = np.where(rng.random(O.NH) < 0.5, -2.0, 2.0)[:, None] * rng.uniform(1.0, 1.5, prm["w1"].shape)
    flat = O.flatten(prm).astype(np.float32)
    X = rng.uniform(-1, 1, (36, n)).astype(np.float32)
    bad = np.arange(0, n, 4)
    X[:, bad] = 3.0e38
    t = MlpTrainer(flat, capacity=512)
    z = t.forward(X)
    t.close()
    ref = _reference(O.unflatten(flat.astype(np.float64)), X.astype(np.float64))
    assert np.isfinite(ref).all()
    # the bounds of the network's other comparisons: a unit at a rounding edge may fall the other way
    err = np.abs(z - ref) / np.maximum(1.0, np.abs(ref))
    assert np.quantile(err, 0.99) <= 1e-4 and err.max() <= 2e-2, (err[bad].max(), err.max())
