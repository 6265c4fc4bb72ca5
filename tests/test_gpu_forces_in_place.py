"""Forces written over the positions they are computed from (F and X one array, or
overlapping ones): every force is that of the positions before the call, bit for
bit, also when a captured graph repeats the call."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import forces_cases as fc  # noqa: E402
from ibamr_amd import structure  # noqa: E402

pytestmark = pytest.mark.gpu


def _ring(n):
    rng = np.random.default_rng(n)
    X = rng.uniform(0.2, 0.8, (n, 3))
    i = rng.permutation(n)   # neighbours far apart in memory
    springs = (i, np.roll(i, 1), rng.uniform(1, 10, n), rng.uniform(0, 1e-3, n))
    beams = (np.roll(i, 1), i, np.roll(i, -1), rng.uniform(0.5, 2.0, n), np.zeros((n, 3)))
    t = np.arange(0, n, 9)
    return 3, X, springs, beams, (t, rng.uniform(1, 10, len(t)), rng.uniform(0, 1, len(t)), X[t] + 1e-3)


@pytest.mark.parametrize("case", ["curve2d", "ring3d", "large"])
@pytest.mark.parametrize("accumulate", [True, False])
@pytest.mark.parametrize("shift", [0, 1])
def test_in_place(orc, case, accumulate, shift):
    ndim, X, springs, beams, targets = _ring(50000) if case == "large" else getattr(fc, case)()
    print("forces in place", case, accumulate, shift, flush=True)
    n = len(X)
    f = structure.Forces(ndim, n, springs, beams, targets)
    buf = torch.full(((n + 1) * ndim,), 0.25, dtype=torch.float64, device="cuda")
    Xd = buf[:n * ndim].view(n, ndim)
    Fd = buf[shift * ndim:(n + shift) * ndim].view(n, ndim)   # one node further: overlapping arrays
    Xd.copy_(torch.from_numpy(X))
    old = Fd.cpu().numpy()
    f.compute(Fd, Xd, accumulate=accumulate)
    want = orc.lagrangian_force(ndim, X, F=old if accumulate else None, springs=springs, beams=beams, targets=targets)
    assert np.array_equal(Fd.cpu().numpy(), want)
    f.close()


def test_captured(orc):
    ndim, X, springs, beams, targets = _ring(3000)
    f = structure.Forces(ndim, len(X), springs, beams, targets)
    Xd = torch.from_numpy(X).cuda()
    F = torch.zeros_like(Xd)
    f.compute(F, Xd)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    with torch.cuda.graph(g, stream=side):
        f.compute(Xd, Xd, accumulate=True, stream=side)
    torch.cuda.synchronize()
    want = X
    for _ in range(3):
        g.replay()
        want = orc.lagrangian_force(ndim, want, F=want, springs=springs, beams=beams, targets=targets)
        assert np.array_equal(Xd.cpu().numpy(), want)
    f.close()
