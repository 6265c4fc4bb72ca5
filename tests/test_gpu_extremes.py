"""FP64 spread on spacings at the ends of the number range, where the reciprocal of dx is
no finite number or few bits of it are left: bit for bit against the oracle (the test
that drops points far from a tile multiplies by that reciprocal)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _dev, _oracle_spread  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["IB_4", "BSPLINE_3", "IB_6"])
@pytest.mark.parametrize("dx", [(1e-310, 1e300), (1e290, 1e-309, 1e15), (1e-70, 1e60, 1e12), (1e-310, 2e-3, 1e302)])
def test_spread_spacings(orc, kernel, dx):
    print("spacings", kernel, dx, flush=True)
    ndim, n = len(dx), 24
    rng = np.random.default_rng(ndim)
    hi = [n * h for h in dx]
    patch = ia.Patch([0] * ndim, [n - 1] * ndim, [0.0] * ndim, hi)
    level = ia.Level(list(dx), [0] * ndim, [n - 1] * ndim, [0.0] * ndim, hi, [0] * ndim, [patch])
    X = np.ascontiguousarray(rng.uniform(0.5, n - 0.5, (300, ndim)) * np.array(dx))
    F = rng.standard_normal(X.shape)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=len(X))
    f = [np.zeros(ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a)) for a in range(ndim)]
    dev = [_dev(a) for a in f]
    plan.bind(0, dev)
    plan.bin(_dev(X))
    plan.spread(0, _dev(F), _dev(X), mode=ia.OVERWRITE)
    want = _oracle_spread(orc, level, plan, f, X, F, kernel)
    assert all(np.count_nonzero(w) > 0 and np.isfinite(w).all() for w in want)
    for a, b in zip(dev, want):
        assert np.array_equal(a.cpu().numpy(), b)
    plan.close()
