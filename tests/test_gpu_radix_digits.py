"""Redistribution's sort at the edges of its tiles (4096 keys), for every digit
width (keys of 8, 9 and 10 bits a pass, one to three passes), and for Lagrangian
indices that are a permutation of 0 .. n-1 (put in order directly) and that are
not (sorted).  The order is exact: patch, cell in box order, Lagrangian index."""
import numpy as np
import pytest
import torch

import ibamr_amd as ia

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,N", [(2, 12), (2, 512), (3, 64), (2, 1024), (3, 128), (3, 384)])
@pytest.mark.parametrize("n", [1, 4096, 4097, 20011])
@pytest.mark.parametrize("lag_kind", ["none", "permutation", "gaps", "one_repeated"])
def test_order(ndim, N, n, lag_kind):
    print("radix digits", ndim, N, n, lag_kind, flush=True)
    rng = np.random.default_rng(7 * ndim + N + n)
    h = 1.0 / N
    lo, hi = [0] * ndim, [N - 1] * ndim
    patch = ia.Patch(lo, hi, [0.0] * ndim, [1.0] * ndim)
    level = ia.Level([h] * ndim, lo, hi, [0.0] * ndim, [1.0] * ndim, [N] * ndim, [patch])
    plan = ia.LevelPlan(level, "IB_4", ia.SIDE, ia.FP64, max_points=n)
    cell = rng.integers(0, N, (n, ndim))
    cell[n // 2:] = rng.integers(0, N, ndim)  # one crowded cell
    X = (cell + 0.5) * h
    lag = rng.permutation(n).astype(np.int32)
    if lag_kind == "gaps":
        lag = (lag.astype(np.int64) * 977).astype(np.int32)
    elif lag_kind == "one_repeated":
        lag[0] = lag[n - 1]
    lin = np.zeros(n, dtype=np.int64)
    for d in range(ndim - 1, -1, -1):
        lin = lin * N + cell[:, d]
    by_lag = np.argsort(lag, kind="stable") if lag_kind != "none" else np.arange(n)
    want = by_lag[np.argsort(lin[by_lag], kind="stable")]
    Xd = torch.from_numpy(X.copy()).cuda()
    lagd = None if lag_kind == "none" else torch.from_numpy(lag).cuda()
    order, poff, _ = plan.redistribute(Xd, lagd)
    assert np.array_equal(order.cpu().numpy(), want)
    assert poff.cpu().tolist() == [0, n]
    assert np.array_equal(Xd.cpu().numpy(), X)
    for depth in (1, 2, 3, 4, 5):
        for dt in (torch.float32, torch.float64):
            src = torch.randn((n, depth), dtype=dt, device="cuda")
            dst = torch.empty_like(src)
            ia.permute_rows(dst, src, order)
            assert torch.equal(dst, src[order.long()])
    plan.close()
