"""Spring networks of so many entries per node that eight lanes share a node's list,
bit for bit against the oracle: a node's entries from none to several rounds of
eight, lists of springs, beams and target points mixed, coincident ends (skipped),
spring laws, the node count at the edge of a workgroup, 2-D and 3-D."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from ibamr_amd import structure  # noqa: E402

pytestmark = pytest.mark.gpu


def _network(ndim, n, rng):
    X = rng.uniform(0.2, 0.8, (n, ndim))
    X[1] = X[0]
    a = np.concatenate([np.zeros(40, int), rng.integers(0, n - 1, 7 * n)])   # node n - 1: target point only
    b = (a + rng.integers(1, n - 1, len(a))) % (n - 1)
    b[0] = 1
    keep = a != b
    a, b = a[keep], b[keep]
    springs = (a, b, rng.uniform(1, 10, len(a)), rng.uniform(0, 0.2, len(a)))
    i = np.arange(1, n - 2)
    beams = (i - 1, i, i + 1, rng.uniform(0.5, 2.0, len(i)), rng.uniform(-1e-3, 1e-3, (len(i), ndim)))
    t = np.arange(n - 1, -1, -5)
    targets = (t, rng.uniform(1, 10, len(t)), rng.uniform(0, 1, len(t)), X[t] + 1e-3)
    return X, springs, beams, targets


def test_long_list_bitwise(orc):
    """Few entries per node on average, but one node of 301."""
    rng = np.random.default_rng(3)
    n = 2000
    X = rng.uniform(0.2, 0.8, (n, 3))
    a = np.concatenate([np.arange(n - 1), np.full(301, 700)])
    b = np.concatenate([np.arange(1, n), np.arange(1000, 1301)])
    springs = (a, b, rng.uniform(1, 10, len(a)), rng.uniform(0, 0.2, len(a)))
    f = structure.Forces(3, n, springs)
    F = torch.full(X.shape, 7.0, dtype=torch.float64, device="cuda")
    f.compute(F, torch.from_numpy(X).cuda())
    assert np.array_equal(F.cpu().numpy(), orc.lagrangian_force(3, X, springs=springs))
    f.close()


@pytest.mark.parametrize("ndim,n", [(2, 32), (2, 33), (3, 64), (3, 65), (3, 4001)])
@pytest.mark.parametrize("laws", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
def test_network_bitwise(orc, ndim, n, laws, accumulate):
    print("force network", ndim, n, laws, accumulate, flush=True)
    rng = np.random.default_rng(n)
    X, springs, beams, targets = _network(ndim, n, rng)
    ns = len(springs[0])
    assert 2 * ns >= 12 * n
    registry = functions = law = None
    if laws:
        idx = rng.choice([0, 2], ns).astype(np.int32)
        off = np.arange(0, 3 * ns + 1, 3).astype(np.int32)
        functions = (idx, off, rng.uniform(0.1, 1.0, 3 * ns))
        registry = {0: structure.SPRING_HOOKEAN, 2: structure.SPRING_POLYNOMIAL}
        law = (np.array([registry[int(k)] for k in idx], dtype=np.int32), off, functions[2])
    U = rng.standard_normal(X.shape)
    F0 = rng.standard_normal(X.shape) if accumulate else np.zeros(X.shape)
    want = orc.lagrangian_force(ndim, X, F=F0, U=U, springs=springs, beams=beams, targets=targets, spring_laws=law)
    f = structure.Forces(ndim, n, springs, beams, targets, registry, functions)
    c = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    F = c(F0) if accumulate else torch.full(X.shape, 7.0, dtype=torch.float64, device="cuda")
    f.compute(F, c(X), c(U), accumulate=accumulate)
    assert np.array_equal(F.cpu().numpy(), want)
    f.close()
