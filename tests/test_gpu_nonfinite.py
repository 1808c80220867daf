"""Infinities, NaN and powers out of range stay with the degrees and the
translations they belong to -- needs an MI355X.  Error measure and bound as in
test_gpu_team.py.
"""
import numpy as np
import pytest

from solidfmm_amd import workload as W
from tests.test_gpu_octet import join
from tests.test_gpu_team import block_errors, run, sfmm  # noqa: F401
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MFMA = 2


# Orders of each team kernel (two, three, four and six chunks per class)
@pytest.mark.parametrize("op", [W.M2M, W.L2L])
@pytest.mark.parametrize("P", [14, 20, 30, 40])
def test_one_sided_degrees(sfmm, orc, op, P):
    """M2M passes a degree on to itself and above, L2L to itself and below:
    an infinity or a NaN in one degree leaves the other side alone, and the
    other translations of its group as they are, bit for bit."""
    n, B = 20, P * (P + 1)
    items, src, dst = physical_batch(orc, op, P, P, n, 17 * P + op)
    zero = np.zeros(len(dst))
    clean = run(sfmm, op, items, src, zero, MFMA if P <= 24 else 0).reshape(n, B)
    want = orc.translate(op, items, src, zero.copy())
    naive = orc.translate(op, items, src, zero.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, zero, items).max(), 1e-13)
    bad = src.copy()
    deg = P - 3 if op == W.M2M else 2
    for i, v in ((3, np.inf), (7, np.nan)):
        bad[int(items["src"][i]) + deg * (deg + 1) + 1] = v
    got = run(sfmm, op, items, bad, zero, MFMA if P <= 24 else 0).reshape(n, B)
    rest = [i for i in range(n) if i not in (3, 7)]
    assert np.array_equal(got[rest], clean[rest])
    keep = slice(0, deg * (deg + 1)) if op == W.M2M else slice((deg + 1) * (deg + 2), B)
    lost = slice(deg * (deg + 1), (deg + 1) * (deg + 2))
    for i in (3, 7):
        w = want.reshape(n, B)[i, keep]
        err = np.linalg.norm(got[i, keep] - w) / np.linalg.norm(w)
        print(f"op {op} P={P} item {i}: {err:.2e} (tol {tol:.2e})", flush=True)
        assert err <= tol
        assert not np.isfinite(got[i, lost]).any()


# A translation of few source degrees beside long ones in its group, at a
# distance whose powers overflow at their degrees
@pytest.mark.parametrize("op", [W.M2M, W.M2L, W.L2L])
def test_powers_beyond_the_degrees(sfmm, orc, op):
    P = 32
    short = physical_batch(orc, op, *((3, P) if op == W.L2L else (2, 30)), 3, 5 + op)
    items = short[0].copy()
    # r^P and r^-P overflow, and no power that a short translation needs does
    r = 1e10 if op == W.L2L else 2e-10
    d = np.sqrt(items["x"] ** 2 + items["y"] ** 2 + items["z"] ** 2)
    for c in "xyz":
        items[c] *= r / d
    # M2L multiplies by up to r^-P: coefficients that keep its results in range
    scale = 1e-220 if op == W.M2L else 1.0
    items, src, nd = join([(items, scale * short[1], short[2]), physical_batch(orc, op, P, P, 13, 9 + op)])
    zero = np.zeros(nd)
    want = orc.translate(op, items, src, zero.copy())
    naive = orc.translate(op, items[3:], src, zero.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, zero, items[3:]).max(), 1e-13)
    got = run(sfmm, op, items, src, zero)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    err = block_errors(got, want, zero, items).max()
    print(f"op {op} P={P}: {err:.2e} (tol {tol:.2e})", flush=True)
    assert err <= tol
