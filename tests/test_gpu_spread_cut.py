"""FP64 spread on a level of more than 2^17 tiles, where the work items' z extent
depends on the kernel (24 values IB_4, IB_6 and BSPLINE_6, 16 the others), on the mode
and on the number of points (IB_4, overwriting): bit for bit against the oracle on
every list that a plan chooses between."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _dev, _oracle_spread  # noqa: E402
from test_gpu_spread_batches import _points  # noqa: E402

pytestmark = pytest.mark.gpu
N = 408


@pytest.mark.parametrize("kernel,npts,modes", [("IB_4", 4000, (ia.OVERWRITE, ia.ACCUMULATE)),
                                               ("IB_4", 300000, (ia.OVERWRITE,)), ("BSPLINE_6", 4000, (ia.OVERWRITE,)),
                                               ("BSPLINE_3", 4000, (ia.OVERWRITE,))])
def test_large_level(orc, kernel, npts, modes):
    print("spread cut", kernel, npts, flush=True)
    rng = np.random.default_rng(npts)
    X = _points(rng, N, 500, npts)
    F = rng.standard_normal(X.shape)
    level = ia.Level.uniform_periodic(N, 3)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=len(X))
    shapes = [ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a) for a in range(3)]
    want = _oracle_spread(orc, level, plan, [np.zeros(s) for s in shapes], X, F, kernel)
    plan.bin(_dev(X))
    for mode in modes:
        # accumulating into zeros: the same values as overwriting anything
        f = [torch.full(s, 0.0 if mode == ia.ACCUMULATE else 3.0, dtype=torch.float64, device="cuda") for s in shapes]
        plan.bind(0, f)
        plan.spread(0, _dev(F), _dev(X), mode=mode)
        for a, b in zip(f, want):
            assert np.array_equal(a.cpu().numpy(), b), mode
    plan.close()


@pytest.mark.parametrize("n,shared", [(40, False), (104, True)])
def test_shapes_with_the_same_pieces(orc, n, shared):
    """8 x 8 x 32 in pieces of 16 and 8 x 8 x 16 are one list: timed once, each accepted
    and reported under its name, the same bits."""
    rng = np.random.default_rng(n)
    X, kernel = _points(rng, n, 300, 2000), "IB_4"
    F = rng.standard_normal(X.shape)
    level = ia.Level.uniform_periodic(n, 3)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=len(X))
    f = [np.zeros(ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a)) for a in range(3)]
    want = _oracle_spread(orc, level, plan, f, X, F, kernel)
    dev = [_dev(a) for a in f]
    plan.bind(0, dev)
    Xd, Fd = _dev(X), _dev(F)
    plan.bin(Xd)
    t = plan.autotune(0, Fd, Xd, reps=2)
    assert sorted(t) == [(8, 8, 16), (8, 8, 32), (16, 4, 32)] and all(v > 0 for v in t.values())
    assert (t[(8, 8, 32)] == t[(8, 8, 16)]) == shared
    assert plan.tile_shape == min(t, key=t.get)
    for sh in t:
        plan.tile_shape = sh
        assert plan.tile_shape == sh
        plan.spread(0, Fd, Xd, mode=ia.OVERWRITE)
        for a, b in zip(dev, want):
            assert np.array_equal(a.cpu().numpy(), b), sh
    plan.close()


@pytest.mark.parametrize("kernel", ["IB_4", "IB_6", "BSPLINE_3"])
def test_tuned_pieces(orc, kernel):
    """Points crowded on a sphere, where pieces of 8 values are the faster ones: the same
    bits after the autotuner's choice, in every mode, with every shape, and again after
    tuning for few points."""
    n, m = 104, 150000
    rng = np.random.default_rng(m)
    D = rng.standard_normal((m, 3))
    X = 0.5 + 0.2 * D / np.linalg.norm(D, axis=1, keepdims=True)
    F = rng.standard_normal(X.shape)
    level = ia.Level.uniform_periodic(n, 3)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=m)
    f = [np.zeros(ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a)) for a in range(3)]
    for k in (m, 100):
        want = _oracle_spread(orc, level, plan, f, X[:k], F[:k], kernel)
        Xd, Fd = _dev(np.ascontiguousarray(X[:k])), _dev(np.ascontiguousarray(F[:k]))
        dev = [_dev(a) for a in f]
        plan.bind(0, dev)
        plan.bin(Xd)
        t = plan.autotune(0, Fd, Xd, reps=2)
        assert t[(8, 8, 16)] == t[(8, 8, 32)] and plan.tile_shape == min(t, key=t.get)
        for sh in t:
            plan.tile_shape = sh
            for mode in (ia.OVERWRITE, ia.ACCUMULATE):
                for a in dev:
                    a.fill_(0.0 if mode == ia.ACCUMULATE else 3.0)
                plan.spread(0, Fd, Xd, mode=mode)
                for a, b in zip(dev, want):
                    assert np.array_equal(a.cpu().numpy(), b), (k, sh, mode)
    plan.close()
