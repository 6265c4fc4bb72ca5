"""2-D spread of few points on levels of 2^14 tiles of 8 x 8 and more, taken in whole
16 x 16 tiles: every mode, stencils over every boundary of a lane's four values, ragged
last tiles, bit for bit against the oracle; and FP32C, in which both tile sizes have to
give the same bits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
import test_gpu_spread_modes as modes  # noqa: E402
from test_gpu_parity import _dev  # noqa: E402
from test_gpu_spread_batches import _points  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ia.OVERWRITE, ia.ACCUMULATE, ia.ACCUMULATE_INTERIOR])
@pytest.mark.parametrize("n,kernel,centering,depth", [
    (1191, "IB_4", ia.SIDE, 1), (1200, "IB_6", ia.SIDE, 1), (1197, "PIECEWISE_LINEAR", ia.SIDE, 1),
    (1194, "BSPLINE_6", ia.SIDE, 1), (1800, "BSPLINE_3", ia.CELL, 1), (560, "BSPLINE_5", ia.CELL, 8)])
def test_few_points_bitwise(orc, mode, n, kernel, centering, depth):
    modes.test_modes_bitwise(orc, mode, 2, n, kernel, centering, depth)


@pytest.mark.parametrize("precision,dtype", [(ia.FP64, torch.float64), (ia.FP32C, torch.float32)])
@pytest.mark.parametrize("kernel", ["PIECEWISE_LINEAR", "IB_4", "BSPLINE_4", "IB_6"])
def test_same_bits_with_many_points(precision, dtype, kernel):
    """Points without force change no sum, but take the spread to tiles of 8 x 8."""
    n = 1003
    rng = np.random.default_rng(n)
    X = _points(rng, n, 700, 3000, 2)
    Y = np.concatenate([X, rng.uniform(0.0, 1.0, (16000, 2))])
    F = np.zeros(Y.shape)
    F[:len(X)] = rng.standard_normal(X.shape)
    F = _dev(F).to(dtype)
    level = ia.Level.uniform_periodic(n, 2)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, precision, max_points=len(Y))
    got = []
    for P in (X, Y):
        f = [torch.full(ia.array_shape(level, 0, plan.data_gcw, ia.SIDE, axis=a), 3.0, dtype=dtype, device="cuda")
             for a in range(2)]
        plan.bind(0, f)
        plan.bin(_dev(P))
        plan.spread(0, F[:len(P)].contiguous(), _dev(P), mode=ia.OVERWRITE)
        got.append([a.cpu().numpy() for a in f])
    for a, b in zip(*got):
        assert np.any(a) and np.array_equal(a, b)
    plan.close()
