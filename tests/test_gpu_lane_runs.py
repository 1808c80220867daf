"""Runs of the lane kernels (items of a wave that share a target) against the
oracle -- needs an MI355X.  Error measure and bound as in test_gpu_octet.py.
"""
import numpy as np
import pytest

from solidfmm_amd import workload as W
from tests.test_gpu_octet import join
from tests.test_gpu_team import block_errors, run, sfmm  # noqa: F401
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LANE, AUTO = 1, 0


def repeated(orc, op, p_in, p_out, n, run_lengths, seed):
    items, src, dst = physical_batch(orc, op, p_in, p_out, n, seed)
    target = np.repeat(np.arange(n), np.resize(run_lengths, n))[:n]
    items["dst"] = target.astype(np.uint64) * np.uint64(p_out * (p_out + 1))
    return items, src, dst


def check(sfmm, orc, op, items, src, nd, family, label):
    want = orc.translate(op, items, src, np.zeros(nd))
    few = items[:200]
    few = few[np.unique(few["dst"], return_index=True)[1]]
    naive = block_errors(orc.translate(op, few, src, np.zeros(nd), naive=True),
                         orc.translate(op, few, src, np.zeros(nd)), np.zeros(nd), few)
    tol = max(20 * naive.max(), 1e-13)
    err = block_errors(run(sfmm, op, items, src, np.zeros(nd), family), want, np.zeros(nd), items).max()
    print(f"{label}: {err:.2e} (tol {tol:.2e})", flush=True)
    assert err <= tol


# One run a wave, eight, nine and more (the tree of shuffles), runs across
# waves, and a last wave that is not full; degrees 7 | 8 change the split
@pytest.mark.parametrize("op", [W.M2M, W.M2L, W.L2L])
@pytest.mark.parametrize("P", [1, 3, 7, 8, 9, 10, 12])
@pytest.mark.parametrize("lengths", [[64], [8], [7], [5, 1, 40, 3, 100, 2]])
def test_lane_runs(sfmm, orc, op, P, lengths):
    parts = [repeated(orc, op, P, P, 64 * 6 + 21, lengths, 5 * P + op)]
    if P > 2:
        parts += [repeated(orc, op, P - 2, P, 64 * 2 + 3, lengths, 6 * P + op)]
        if op != W.L2L:
            parts += [repeated(orc, op, P, P - 1, 64 * 2 + 7, lengths, 7 * P + op)]
    parts += [repeated(orc, op, 1, 1, 10, [10], 1)]
    items, src, nd = join(parts)
    if op != W.M2L:
        for c in "xyz":
            items[c][130:200:13] = 0.0
    check(sfmm, orc, op, items, src, nd, LANE, f"op {op} P={P} runs {lengths}")


@pytest.mark.parametrize("P", [8, 12])
@pytest.mark.parametrize("n", [39000, 41000])
def test_default_on_repeated_targets(sfmm, orc, P, n):
    """Both sides of the item count from which lanes take repeated targets."""
    parts = [repeated(orc, W.M2L, P, P, 300, [50], P), repeated(orc, W.M2L, 1, P, n - 300, [90], P + 1)]
    items, src, nd = join(parts)
    check(sfmm, orc, W.M2L, items, src, nd, AUTO, f"default P={P} n={n}")


# Lists long enough for the sums through LDS: waves of one run, of a few, and
# of more than the LDS sums take; runs across waves; a last wave that is not full
@pytest.mark.parametrize("op", [W.M2M, W.M2L, W.L2L])
@pytest.mark.parametrize("P", [1, 3, 7, 8, 9, 12])
def test_long_lists_of_long_runs(sfmm, orc, op, P):
    parts = [repeated(orc, op, P, P, 64 * 4 + 21, lengths, 5 * P + op)
             for lengths in ([64], [20], [13, 12, 13], [3, 1, 40, 2, 100, 2])]
    parts += [repeated(orc, op, 1, P, 66000, [64], P)]
    items, src, nd = join(parts)
    if op != W.M2L:
        for c in "xyz":
            items[c][130:200:13] = 0.0
    check(sfmm, orc, op, items, src, nd, LANE, f"op {op} P={P}")
