"""FP64 spread in batches of hits (k_spread3b) where the batching can go wrong,
bit for bit against the oracle (the order of summation does not depend on the
batches): bins of more than 64 points beside bins of a few (batch ends inside a
bin, never inside a 64-point chunk), every z extent of the work items (8 below
4096 tiles, 24 from 2^17 on, 16 between), spacings whose cell volume is no power
of two (quotients from reciprocals), tiny, zero and infinite forces.  The same
for the 2-D kernel (k_spread2: 8 x 8 tiles, batches of any 64 points)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _dev, _oracle_spread  # noqa: E402

pytestmark = pytest.mark.gpu


def _check(orc, n, kernel, X, F, mode=ia.OVERWRITE):
    print("batches", n, kernel, X.shape[0], flush=True)
    ndim = X.shape[1]
    level = ia.Level.uniform_periodic(n, ndim)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=X.shape[0])
    f = [np.zeros(ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a)) for a in range(ndim)]
    dev = [_dev(a) for a in f]
    plan.bind(0, dev)
    plan.bin(_dev(X))
    plan.spread(0, _dev(F), _dev(X), mode=mode)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        want = _oracle_spread(orc, level, plan, f, X, F, kernel)
    for a, b in zip(dev, want):
        assert np.array_equal(a.cpu().numpy(), b, equal_nan=True)
    plan.close()


def _points(rng, n, dense, sparse, ndim=3):
    """dense points in two cells' worth of space across a bin corner and on the
    periodic edge, sparse ones anywhere."""
    h = 1.0 / n
    X = rng.uniform(0.0, 1.0, (sparse, ndim))
    c = 8 * h * rng.integers(1, max(2, n // 8 - 1), ndim)
    D = np.remainder(c + rng.uniform(-1.2 * h, 1.2 * h, (dense, ndim)), 1.0)
    E = np.remainder(rng.uniform(-2 * h, 2 * h, (dense // 2, ndim)), 1.0)
    return np.concatenate([X, D, E])


@pytest.mark.parametrize("n,kernel", [(24, "IB_6"), (40, "IB_4"), (37, "BSPLINE_3"), (33, "PIECEWISE_LINEAR"),
                                      (40, "BSPLINE_5"), (104, "IB_6"), (107, "BSPLINE_3"), (112, "BSPLINE_4")])
def test_batches_bitwise(orc, n, kernel):
    rng = np.random.default_rng(n)
    X = _points(rng, n, 700, 5000)
    _check(orc, n, kernel, X, rng.standard_normal(X.shape))


@pytest.mark.parametrize("n,kernel", [(24, "IB_6"), (40, "IB_4"), (37, "BSPLINE_3"), (130, "PIECEWISE_LINEAR"),
                                      (33, "BSPLINE_5"), (48, "BSPLINE_6")])
def test_2d_bitwise(orc, n, kernel):
    rng = np.random.default_rng(n)
    X = _points(rng, n, 700, 2000, 2)
    F = rng.standard_normal(X.shape)
    F[:20] *= 1e-200
    F[20:30] = 0.0
    F[30] = np.inf
    _check(orc, n, kernel, X, F)


def test_24_values(orc):
    rng = np.random.default_rng(5)
    X = _points(rng, 408, 900, 6000)
    _check(orc, 408, "IB_4", X, rng.standard_normal(X.shape))


@pytest.mark.parametrize("kernel", ["IB_4", "BSPLINE_3"])
def test_extreme_forces(orc, kernel):
    rng = np.random.default_rng(7)
    X = rng.uniform(0.0, 1.0, (400, 3))
    X[:8] = np.array([0.0, 0.25, 0.5])   # on cell faces: weights of exactly zero
    F = rng.standard_normal(X.shape)
    F[10:40] *= 1e-290
    F[40:60] *= 1e250
    F[60:80] = 0.0
    F[80] = np.inf
    F[81] = np.nan
    _check(orc, 36, kernel, X, F)
