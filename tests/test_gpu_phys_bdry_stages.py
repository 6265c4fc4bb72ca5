"""Physical boundary operators run in stages (operators of one component whose
regions do not meet run together): patches so thin that opposite faces' regions
meet, domains with one walled axis pair left periodic, one patch with all 26
boundary pieces, against the oracle's sequence of operators, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import ibamr_amd as ia  # noqa: E402
from test_gpu_parity import _dev  # noqa: E402
from test_gpu_phys_bdry import _boxes_and_coefs, _level  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,side,depth,cuts,periodic", [
    (10, True, 1, None, ()), (10, False, 3, None, ()), (9, True, 1, [[4], [5], [3, 6]], ()),
    (12, False, 1, [[4], [8], [5]], ()), (9, True, 1, [[4], [], []], (1,)), (5, True, 1, None, ()),
    (5, False, 2, None, (0,))])
@pytest.mark.parametrize("adjoint", [True, False])
def test_stages_match_oracle(orc, n, side, depth, cuts, periodic, adjoint):
    print("bdry stages", n, side, depth, cuts, periodic, adjoint, flush=True)
    gcw = 3
    level = _level(3, n, cuts, periodic)
    plan = ia.LevelPlan(level, "IB_4", ia.SIDE if side else ia.CELL, ia.FP64, depth=depth, data_gcw=[gcw] * 3,
                        max_points=1)
    rng = np.random.default_rng(n * 10 + side)
    narr = 3 if side else depth
    boxes, abg = _boxes_and_coefs(level, gcw, narr, rng)
    plan.set_physical_boundary(boxes, abg)
    plan.set_physical_boundary(boxes, abg)   # replacing the tables
    per = 3 if side else 1
    arrays = [rng.standard_normal(ia.array_shape(level, p, [gcw] * 3, plan.centering, axis=a, depth=depth))
              for p in range(len(level.patches)) for a in range(per)]
    dev = [_dev(a) for a in arrays]
    plan.bind(0, dev)
    if adjoint:
        plan.accumulate_physical_boundary(0)
    else:
        plan.fill_physical_boundary(0)
    torch.cuda.synchronize()
    for p, P in enumerate(level.patches):
        own = [k for k, b in enumerate(boxes) if b[0] == p]
        ref = [arrays[p * per + a].copy() for a in range(per)]
        orc.phys_bdry(ref, P.ilower, P.iupper, gcw, level.dx, [boxes[k][1:] for k in own], abg[own], side, adjoint,
                      depth=depth)
        for a in range(per):
            assert np.array_equal(dev[p * per + a].cpu().numpy(), ref[a]), (p, a)
    plan.close()
