"""The right-hand side kernel with 1, 2 and 8 lanes per node, bit for bit against
the oracle: meshes of more nodes than 8 lanes each fill the GPU with (chains of
EDGE2 elements: 1 lane with 2 points per element, 2 lanes with 5), and small ones
of 8 lanes whose nodes have from no entry to more than two rounds of entries."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402

pytestmark = pytest.mark.gpu


def _chain(n, rng):
    i = rng.permutation(n).astype(np.int32)
    return np.stack([i[:-1], i[1:]], axis=1)


def _fans(n, rng):
    """Triangles that share node 0, 1 or 2 with 9, 17 and 30 of them; nodes from n - 5 on unused."""
    e = [[c, *rng.choice(np.arange(3, n - 5), 2, replace=False)] for c, m in ((0, 9), (1, 17), (2, 30)) for _ in range(m)]
    return np.array(e, dtype=np.int32)[rng.permutation(len(e))]


@pytest.mark.parametrize("mesh,nnodes,nqp", [("chain", 65537, 2), ("chain", 65537, 5), ("chain", 70001, 9),
                                             ("chain", 65536, 2), ("fans", 40, 1), ("fans", 41, 4)])
@pytest.mark.parametrize("nvars", [1, 3, 8])
def test_lanes_bitwise(orc, mesh, nnodes, nqp, nvars):
    print("fe rhs lanes", mesh, nnodes, nqp, nvars, flush=True)
    rng = np.random.default_rng(nnodes + nqp)
    E = _chain(nnodes, rng) if mesh == "chain" else _fans(nnodes, rng)
    phi = rng.standard_normal((E.shape[1], nqp))
    J = rng.uniform(0.5, 1.5, (len(E), nqp))
    m = ia.FEMesh(E, nnodes)
    c = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for dt in (np.float64, np.float32):
        U = rng.standard_normal((len(E) * nqp, nvars)).astype(dt)
        F = torch.full((nnodes, nvars), 7.0, dtype=torch.float64, device="cuda")
        m.integrate_rhs(F, c(U), c(phi), c(J))
        assert np.array_equal(F.cpu().numpy(), orc.fe_integrate_rhs(E, phi, J, U.astype(np.float64), nnodes))
        old = rng.standard_normal((nnodes, nvars))
        F = c(old)
        m.integrate_rhs(F, c(U), c(phi), c(J), accumulate=True)
        assert np.array_equal(F.cpu().numpy(), orc.fe_integrate_rhs(E, phi, J, U.astype(np.float64), nnodes, F=old))
    m.close()
