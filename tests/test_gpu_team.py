"""Team kernels (several waves per group of translations) against the oracle
-- needs an MI355X.

All run on physical (decaying) expansions.  Error measure: per
item, the 2-norm of the difference over the 2-norm of the oracle's block.
Bound: 20 times the largest distance of the oracle from the naive O(P^4)
formulas on the same items (two evaluations of one algorithm, whose errors
sit at that distance), and not below 1e-13.
"""
import numpy as np
import pytest

from solidfmm_amd import workload as W
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

OPS = [W.M2M, W.M2L, W.L2L]


@pytest.fixture(scope="module")
def sfmm():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    import solidfmm_amd
    solidfmm_amd.load()
    return solidfmm_amd


def run(sfmm, op, items, src, dst0, family=0):
    ctx = sfmm.Context(int(max(items["p_in"].max(), items["p_out"].max())))
    ctx.set_kernels(family)
    plan = sfmm.Plan(ctx, op, items)
    s, d = torch.from_numpy(src).to("cuda"), torch.from_numpy(dst0.copy()).to("cuda")
    plan.execute(s, d)
    torch.cuda.synchronize()
    return d.cpu().numpy()


def block_errors(got, want, dst0, items):
    """Per distinct target: |got - want| / |want - dst0|."""
    out = []
    for off, p in sorted({(int(o), int(p)) for o, p in zip(items["dst"], items["p_out"])}):
        sl = slice(off, off + p * (p + 1))
        scale = np.linalg.norm(want[sl] - dst0[sl])
        d = np.linalg.norm(got[sl] - want[sl])
        out.append(d / scale if scale else (np.inf if d else 0.0))
    return np.array(out)


def check(sfmm, orc, op, items, src, dst0, label):
    want = orc.translate(op, items, src, dst0.copy())
    naive = orc.translate(op, items, src, dst0.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, dst0, items).max(), 1e-13)
    err = block_errors(run(sfmm, op, items, src, dst0), want, dst0, items).max()
    print(f"{label}: {err:.2e} (tol {tol:.2e})", flush=True)
    assert err <= tol


# 25 and 32: ends of the kernel with four chunks per parity class; 33: the
# next one; 36 and 48: 8 translations per workgroup and the largest triangle
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("P,n", [(25, 1), (25, 17), (31, 15), (32, 16), (32, 33), (33, 9), (36, 8), (36, 17),
                                 (41, 5), (47, 9), (48, 3)])
def test_high_orders_square(sfmm, orc, op, P, n):
    items, src, dst = physical_batch(orc, op, P, P, n, 7 * P + n + op)
    dst0 = 1e-3 * np.resize(src, len(dst))  # targets are added to
    check(sfmm, orc, op, items, src, dst0, f"op {op} P={P} n={n}")


@pytest.mark.parametrize("op", OPS)
def test_high_orders_mixed(sfmm, orc, op):
    """One list of order pairs up to 48 (and one above, and one below 25),
    zero shifts among them, in shuffled order."""
    pairs = [(25, 25), (30, 26), (26, 31), (32, 3), (2, 32), (33, 33), (48, 34), (35, 48), (1, 40), (45, 1), (50, 49),
             (24, 20)]
    if op == W.L2L:  # truncation beyond p_out + 1 is covered against the naive formula only
        pairs = [(a, b) for a, b in pairs if a <= b + 1] + [(27, 26), (41, 40)]
    rng = np.random.default_rng(11 + op)
    parts = [physical_batch(orc, op, a, b, 5, 100 + 10 * a + b + op) for a, b in pairs]
    so = np.cumsum([0] + [len(p[1]) for p in parts])
    do = np.cumsum([0] + [len(p[2]) for p in parts])
    items = []
    for k, (it, _, _) in enumerate(parts):
        it = it.copy()
        it["src"] += np.uint64(so[k])
        it["dst"] += np.uint64(do[k])
        if op != W.M2L:
            for c in "xyz":
                it[c][k % 5] = 0.0
        items.append(it)
    items = rng.permutation(np.concatenate(items))
    src = np.concatenate([p[1] for p in parts])
    check(sfmm, orc, op, items, src, np.zeros(do[-1]), f"mixed op {op}")


@pytest.mark.parametrize("P", [26, 40])
def test_high_orders_repeated_targets(sfmm, orc, P):
    """Targets repeated often enough for scratch blocks and a reduction."""
    items, src, dst = physical_batch(orc, W.M2L, P, P, 29, 3 * P)
    items["dst"] = (np.arange(29) % 4) * P * (P + 1)
    check(sfmm, orc, W.M2L, items, src, np.zeros(len(dst)), f"repeated P={P}")


# Short lists up to order 24, where plans choose between lanes, team and
# straight-line kernels: orders around 8 chunks' ends (9, 17, 24), 20 | 21 as
# the last straight-line order, item counts around a group of 16, around 256
# groups (eight waves a group, then four) and around the dispatch's 4,096
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("P,n", [(8, 1), (8, 4096), (8, 4097), (9, 15), (11, 17), (12, 33), (15, 16), (16, 17),
                                 (16, 4097), (17, 31), (18, 4113), (20, 16), (21, 49), (24, 18)])
def test_low_orders_square(sfmm, orc, op, P, n):
    items, src, dst = physical_batch(orc, op, P, P, n, 7 * P + n + op)
    dst0 = 1e-3 * np.resize(src, len(dst))
    check(sfmm, orc, op, items, src, dst0, f"op {op} P={P} n={n}")


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("family", [0, 2])
def test_low_orders_mixed(sfmm, orc, op, family):
    """Order pairs up to 24, zero shifts among them, each target three times
    in a row (rounds) or eleven times (scratch blocks and runs)."""
    pairs = [(1, 1), (1, 9), (8, 3), (8, 8), (9, 10), (11, 2), (12, 13), (16, 16), (16, 17), (17, 5), (20, 20),
             (21, 20), (19, 24), (24, 1)]
    if op == W.L2L:
        pairs = [(a, b) for a, b in pairs if a <= b + 1]
    rng = np.random.default_rng(23 + op)
    for repeats in (3, 11):
        items, srcs, so, do = [], [], 0, 0
        for a, b in pairs:
            it, s, d = physical_batch(orc, op, a, b, 2 * repeats, 300 + 10 * a + b + op)
            it = it.copy()
            it["src"] += np.uint64(so)
            it["dst"] = np.uint64(do) + np.arange(2 * repeats, dtype=np.uint64) % 2 * np.uint64(b * (b + 1))
            if op != W.M2L:
                for c in "xyz":
                    it[c][a % 5] = 0.0
            items.append(it)
            srcs.append(s)
            so, do = so + len(s), do + len(d)
        items = rng.permutation(np.concatenate(items))
        src = np.concatenate(srcs)
        want = orc.translate(op, items, src, np.zeros(do))
        naive = orc.translate(op, items, src, np.zeros(do), naive=True)
        tol = max(20 * block_errors(naive, want, np.zeros(do), items).max(), 1e-13)
        err = block_errors(run(sfmm, op, items, src, np.zeros(do), family), want, np.zeros(do), items).max()
        print(f"mixed op {op} family {family} repeats {repeats}: {err:.2e} (tol {tol:.2e})", flush=True)
        assert err <= tol


@pytest.mark.parametrize("op", OPS)
def test_forced_generic_kernel(sfmm, orc, op):
    """A context that asks for the generic family gets one launch of the
    one-workgroup kernel for all orders; the default has the team kernels for
    25 to 32 and for 33 to 48."""
    parts = [physical_batch(orc, op, P, P, 5, 13 * P + op) for P in (20, 27, 36)]
    items, src, off = [], [], [0, 0]
    for it, s, d in parts:
        it = it.copy()
        it["src"] += np.uint64(off[0])
        it["dst"] += np.uint64(off[1])
        items.append(it)
        src.append(s)
        off = [off[0] + len(s), off[1] + len(d)]
    items, src, zero = np.concatenate(items), np.concatenate(src), np.zeros(off[1])
    for family, launches in ((0, 3), (3, 1)):
        ctx = sfmm.Context(36)
        ctx.set_kernels(family)
        info = sfmm.Plan(ctx, op, items).launch_info()
        assert len(info) == launches, info
    want = orc.translate(op, items, src, zero.copy())
    naive = orc.translate(op, items, src, zero.copy(), naive=True)
    tol = max(20 * block_errors(naive, want, zero, items).max(), 1e-13)
    assert block_errors(run(sfmm, op, items, src, zero, 3), want, zero, items).max() <= tol


@pytest.mark.parametrize("op,P", [(W.M2L, 28), (W.M2L, 36), (W.M2M, 32)])
def test_high_orders_truth(sfmm, orc, op, P):
    """Against the binary128 evaluation: the median over the items of the
    largest degree's error (M2M: of the block's) is no larger than the
    oracle's, whose powers are products of one factor at a time.  Medians of
    360 items scatter by 5 %."""
    import math

    import oracle
    truth, n = oracle.Truth(), 120
    ours, theirs = [], []
    for seed in (1, 2, 3):
        items, src, dst = W.uniform_batch(op, P, P, n, seed, shift="m2l" if op == W.M2L else "octant")
        s = src.reshape(n, -1)
        for k in range(P):  # decaying coefficients
            s[:, k * (k + 1):(k + 1) * (k + 2)] *= 0.8 ** k / math.factorial(k)
        zero = np.zeros(len(dst))
        want = np.asarray(truth.translate(op, items, src, len(dst), dst0=zero)[0], dtype=np.float64)
        for out, got in ((ours, run(sfmm, op, items, src, zero)), (theirs, orc.translate(op, items, src, zero.copy()))):
            if op == W.M2L:
                out.append(oracle.degree_errors(got, want, P).max(axis=1))
            else:
                d, w = (got - want).reshape(n, -1), want.reshape(n, -1)
                out.append(np.linalg.norm(d, axis=1) / np.linalg.norm(w, axis=1))
    a, b = np.median(np.concatenate(ours)), np.median(np.concatenate(theirs))
    print(f"op {op} P={P}: median {a:.2e}, oracle {b:.2e}", flush=True)
    assert a <= 1.05 * b
