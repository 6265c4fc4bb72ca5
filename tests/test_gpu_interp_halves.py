"""FP64 interpolation from whole and from halved superbins on both sides of the
rules that choose (125 superbins: halves; 216: halves, BSPLINE_6 by the points; 343:
by the points, which fill more than 256 superbins, or a part of the level only; 4913:
whole ones), bit for bit against
the oracle: points on superbin and half-superbin faces, crowded cells, a level of
one patch and one whose superbins several patches share."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _arrays, _dev, _oracle_interp, _periodic_fill_np  # noqa: E402

pytestmark = pytest.mark.gpu


def _points(rng, n, part=1.0):
    h = 1.0 / n
    X = rng.uniform(0.0, 1.0, (3000, 3)) * [1.0, 1.0, part]
    D = 0.5 + h * rng.uniform(-1.0, 1.0, (700, 3))
    E = rng.uniform(0.0, 1.0, (300, 3))
    E[:, 2] = 8 * h * rng.integers(0, int(part * n) // 8, 300) + rng.choice([-1e-12, 0.0, 1e-12], 300)
    return np.ascontiguousarray(np.clip(np.concatenate([X, D, E]), 0.0, np.nextafter(1.0, 0.0)))


@pytest.mark.parametrize("n,part", [(80, 1.0), (88, 1.0), (88, 0.4), (104, 1.0), (104, 0.4)])
@pytest.mark.parametrize("kernel", ["IB_4", "IB_6", "BSPLINE_3", "BSPLINE_5", "BSPLINE_6", "PIECEWISE_LINEAR"])
def test_one_patch(orc, n, part, kernel):
    print("interp halves", n, part, kernel, flush=True)
    rng = np.random.default_rng(n)
    level = ia.Level.uniform_periodic(n, 3)
    X = _points(rng, n, part)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=len(X))
    u = [_periodic_fill_np(a, plan.data_gcw[0], n) for a in _arrays(level, plan, rng)]
    plan.bind(0, [_dev(a) for a in u])
    plan.bin(_dev(X))
    U = torch.full((len(X), 3), float("nan"), dtype=torch.float64, device="cuda")
    plan.interp(0, U, _dev(X))
    assert np.array_equal(U.cpu().numpy(), _oracle_interp(orc, level, plan, u, X, kernel))
    plan.close()


def test_more_superbins(orc):
    test_one_patch(orc, 260, 1.0, "IB_4")


def test_binned_again(orc):
    """One plan, points that fill the level, then a part of it, in turn: each
    binning counts anew."""
    n, kernel = 104, "BSPLINE_3"
    rng = np.random.default_rng(7)
    level = ia.Level.uniform_periodic(n, 3)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=4000)
    u = [_periodic_fill_np(a, plan.data_gcw[0], n) for a in _arrays(level, plan, rng)]
    plan.bind(0, [_dev(a) for a in u])
    for part in (1.0, 0.3, 1.0, 0.1):
        X = _points(rng, n, part)
        plan.bin(_dev(X))
        U = torch.full((len(X), 3), float("nan"), dtype=torch.float64, device="cuda")
        plan.interp(0, U, _dev(X))
        assert np.array_equal(U.cpu().numpy(), _oracle_interp(orc, level, plan, u, X, kernel))
    plan.close()


@pytest.mark.parametrize("n", [80, 88, 104])
@pytest.mark.parametrize("kernel", ["IB_4", "BSPLINE_3"])
def test_shared_superbins(orc, n, kernel):
    """Patches cut inside superbins: every point from the patch that owns its cell."""
    print("interp halves, patches", n, kernel, flush=True)
    rng = np.random.default_rng(n + 1)
    h = 1.0 / n
    cuts = [[0, 27, n], [0, 40, n], [0, 12, 43, n]]
    patches = []
    for k in range(3):
        for j in range(2):
            for i in range(2):
                lo = [cuts[0][i], cuts[1][j], cuts[2][k]]
                hi = [cuts[0][i + 1] - 1, cuts[1][j + 1] - 1, cuts[2][k + 1] - 1]
                patches.append(ia.Patch(lo, hi, [v * h for v in lo], [(v + 1) * h for v in hi]))
    level = ia.Level([h] * 3, [0] * 3, [n - 1] * 3, [0.0] * 3, [1.0] * 3, [n] * 3, patches)
    X = _points(rng, n)
    plan = ia.LevelPlan(level, kernel, ia.SIDE, ia.FP64, max_points=len(X))
    u = [_dev(a) for a in _arrays(level, plan, rng)]
    plan.bind(0, u)
    plan.fill_ghosts(0)
    plan.bin(_dev(X))
    U = torch.full((len(X), 3), float("nan"), dtype=torch.float64, device="cuda")
    plan.interp(0, U, _dev(X))
    torch.cuda.synchronize()
    want = _oracle_interp(orc, level, plan, [a.cpu().numpy() for a in u], X, kernel)
    assert np.array_equal(U.cpu().numpy(), want)
    plan.close()
