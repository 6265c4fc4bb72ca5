"""FP64 spread in every mode over arrays that hold values, bit for bit against the
oracle, in 2-D and 3-D: crowded bins beside sparse ones, spacings whose cell volume
is a power of two (exact products by its reciprocal) and is not (corrected
quotients), every kernel width; cell data of several components."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _arrays, _dev, _oracle_spread  # noqa: E402
from test_gpu_spread_batches import _points  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ia.OVERWRITE, ia.ACCUMULATE, ia.ACCUMULATE_INTERIOR])
@pytest.mark.parametrize("ndim,n,kernel,centering,depth", [
    (3, 32, "BSPLINE_3", ia.SIDE, 1), (3, 32, "PIECEWISE_LINEAR", ia.SIDE, 1), (3, 37, "BSPLINE_5", ia.SIDE, 1),
    (3, 64, "BSPLINE_6", ia.SIDE, 1), (3, 30, "IB_6", ia.SIDE, 1), (3, 32, "BSPLINE_4", ia.CELL, 3),
    (3, 35, "IB_4", ia.CELL, 2), (2, 64, "BSPLINE_3", ia.SIDE, 1), (2, 32, "PIECEWISE_LINEAR", ia.CELL, 2),
    (2, 50, "IB_4", ia.SIDE, 1), (2, 41, "BSPLINE_6", ia.CELL, 3)])
def test_modes_bitwise(orc, mode, ndim, n, kernel, centering, depth):
    print("spread modes", mode, ndim, n, kernel, centering, depth, flush=True)
    rng = np.random.default_rng(n)
    X = _points(rng, n, 700, 3000, ndim)
    level = ia.Level.uniform_periodic(n, ndim)
    plan = ia.LevelPlan(level, kernel, centering, ia.FP64, depth=depth, max_points=len(X))
    F = rng.standard_normal((len(X), ndim if centering == ia.SIDE else depth))
    old = _arrays(level, plan, rng)
    dev = [_dev(a) for a in old]
    plan.bind(0, dev)
    plan.bin(_dev(X))
    plan.spread(0, _dev(F), _dev(X), mode=mode)
    torch.cuda.synchronize()
    zero = [np.zeros_like(a) for a in old]
    want = _oracle_spread(orc, level, plan, old if mode == ia.ACCUMULATE else zero, X, F, kernel)
    for a, (got, w, o) in enumerate(zip(dev, want, old)):
        got = got.cpu().numpy()
        if mode != ia.ACCUMULATE_INTERIOR:
            assert np.array_equal(got, w), a
            continue
        inner = tuple(slice(g, -g) for g in reversed(plan.data_gcw))
        if centering == ia.CELL:
            inner = (slice(None),) + inner
        ref = o.copy()
        ref[inner] = o[inner] + w[inner]
        assert np.array_equal(got, ref), a
    plan.close()
