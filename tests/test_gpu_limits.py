"""Both sides of the list lengths at which plans change kernels -- needs an
MI355X.  Error measure and bound as in test_gpu_octet.py.
"""
import numpy as np
import pytest

from solidfmm_amd import workload as W
from tests.test_gpu_lane_runs import check, repeated
from tests.test_gpu_octet import join
from tests.test_gpu_team import block_errors, sfmm  # noqa: F401
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

AUTO, LANE, MFMA = 0, 1, 2


# Lists of n items, most of them of order 1 -> P, in runs of 16 and more: a
# run that the plan lays out for 16 translations a group and the launch for 8
# (or the other way round) loses part of its sum
@pytest.mark.parametrize("op,P,limit", [(W.M2M, 9, 4096), (W.M2L, 13, 4096), (W.L2L, 10, 4096), (W.M2L, 16, 8192),
                                        (W.M2M, 19, 12288), (W.M2L, 20, 24576), (W.M2L, 22, 32768)])
@pytest.mark.parametrize("more", [0, 1])
def test_runs_at_the_team_limit(sfmm, orc, op, P, limit, more):
    n = limit + more
    parts = [repeated(orc, op, P, P, 50, [16, 17, 3], P), repeated(orc, op, 1, P, n - 50, [16, 40, 1], P + 1)]
    items, src, nd = join(parts)
    check(sfmm, orc, op, items, src, nd, MFMA, f"op {op} P={P} n={n}")


@pytest.mark.parametrize("P,n,family", [(9, 8192, MFMA), (9, 8193, LANE), (9, 16384, LANE), (9, 16385, MFMA),
                                        (9, 24577, LANE), (9, 32769, MFMA), (10, 8193, LANE), (10, 24577, MFMA),
                                        (11, 16384, LANE), (11, 16385, MFMA), (8, 8193, MFMA), (12, 8193, MFMA)])
def test_l2l_default(sfmm, orc, P, n, family):
    """L2L of orders 9 to 11 stays on lanes where octets fill a step badly."""
    items, src, dst = physical_batch(orc, W.L2L, P, P, n, P + n)
    ctx = sfmm.Context(P)
    plan = sfmm.Plan(ctx, W.L2L, items)
    assert [i[0] for i in plan.launch_info()] == [family]
    d = torch.zeros(len(dst), dtype=torch.float64, device="cuda")
    plan.execute(torch.from_numpy(src).to("cuda"), d)
    torch.cuda.synchronize()
    want = orc.translate(W.L2L, items, src, np.zeros(len(dst)))
    few = items[:200]
    zero = np.zeros(len(dst))
    naive = orc.translate(W.L2L, few, src, zero.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, zero, few).max(), 1e-13)
    assert block_errors(d.cpu().numpy(), want, zero, items).max() <= tol


# Repeated targets: lanes for long lists of long runs, by their mean length
# and not by the one target that repeats most
@pytest.mark.parametrize("op,P,n,lengths,family", [
    (W.M2L, 12, 70000, [5] + [1] * 69995, MFMA),   # one target of five items
    (W.M2L, 12, 70000, [40], MFMA), (W.M2M, 10, 70000, [8], MFMA), (W.L2L, 8, 110000, [64], MFMA),
    (W.M2L, 8, 110000, [64], LANE), (W.M2M, 9, 110000, [40], LANE), (W.M2L, 9, 50000, [64], LANE),
    (W.M2L, 9, 66000, [20], MFMA), (W.M2M, 9, 50000, [64], MFMA), (W.M2L, 11, 110000, [64], MFMA)])
def test_repeated_targets_default(sfmm, orc, op, P, n, lengths, family):
    parts = [repeated(orc, op, P, P, 50, [16, 17, 3], P), repeated(orc, op, 1, P, n - 50, lengths, P + 1)]
    items, src, nd = join(parts)
    info = sfmm.Plan(sfmm.Context(P), op, items).launch_info()
    assert [i[0] for i in info] == [family], info
    check(sfmm, orc, op, items, src, nd, AUTO, f"op {op} P={P} n={n}")


@pytest.mark.parametrize("P,n,family", [(9, 8192, MFMA), (9, 20000, LANE), (10, 30000, LANE), (11, 17000, LANE),
                                        (8, 20000, MFMA), (12, 20000, MFMA)])
def test_l2l_of_children_default(sfmm, orc, P, n, family):
    """L2L from parents of eight children, orders 9 to 11, stays on lanes."""
    items, src, dst = physical_batch(orc, W.L2L, P, P, n, P + n)
    items["src"] = items["src"][np.arange(n) // 8]
    ctx = sfmm.Context(P)
    plan = sfmm.Plan(ctx, W.L2L, items)
    assert [i[0] for i in plan.launch_info()] == [family]
    zero = np.zeros(len(dst))
    d = torch.zeros(len(dst), dtype=torch.float64, device="cuda")
    plan.execute(torch.from_numpy(src).to("cuda"), d)
    torch.cuda.synchronize()
    want = orc.translate(W.L2L, items, src, zero.copy())
    naive = orc.translate(W.L2L, items[:200], src, zero.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, zero, items[:200]).max(), 1e-13)
    assert block_errors(d.cpu().numpy(), want, zero, items).max() <= tol
