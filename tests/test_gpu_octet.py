"""Octet kernels (a wave per eight translations) against the oracle -- needs
an MI355X.  Lists are longer than the team kernels take, so most of their
items are cheap ones of orders (P, 1) or (1, P).

Error measure and bound as in test_gpu_team.py, the distance of the oracle
from the naive O(P^4) formulas taken over the first 200 items.
"""
import numpy as np
import pytest

from solidfmm_amd import workload as W
from tests.test_gpu_team import block_errors, run, sfmm  # noqa: F401
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

OPS = [W.M2M, W.M2L, W.L2L]
MFMA = 2


def join(parts):
    """One list of several batches, each on pool ranges of its own."""
    items, srcs, so, do = [], [], 0, 0
    for it, s, d in parts:
        it = it.copy()
        it["src"] += np.uint64(so)
        it["dst"] += np.uint64(do)
        items.append(it)
        srcs.append(s)
        so, do = so + len(s), do + len(d)
    return np.concatenate(items), np.concatenate(srcs), do


def check(sfmm, orc, op, items, src, dst0, label):
    want = orc.translate(op, items, src, dst0.copy())
    few = items[:200]
    few = few[np.unique(few["dst"], return_index=True)[1]]
    naive = block_errors(orc.translate(op, few, src, dst0.copy(), naive=True),
                         orc.translate(op, few, src, dst0.copy()), dst0, few)
    tol = max(20 * naive.max(), 1e-13)
    err = block_errors(run(sfmm, op, items, src, dst0, MFMA), want, dst0, items).max()
    print(f"{label}: {err:.2e} (tol {tol:.2e})", flush=True)
    assert err <= tol


# Ends of the chunk counts (8 | 9, 16 | 17, 24), of the registers' variants
# (12 | 13, 14 | 15) and of the dispatch (M2L 22); the list ends inside a
# group (37 = 4 groups and 5)
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("P", [1, 2, 5, 8, 9, 12, 13, 14, 15, 16, 17, 20, 21, 22, 24])
def test_octet_orders(sfmm, orc, op, P):
    """Square items, every smaller order against P, zero shifts, in one list."""
    parts = [physical_batch(orc, op, P, P, 37, 5 * P + op)]
    for a in range(1, P):
        parts += [physical_batch(orc, op, a, P, 2, 31 * a + P + op)]
        if op != W.L2L:
            parts += [physical_batch(orc, op, P, a, 2, 37 * a + P + op)]
    n = 12800 if P > 18 else 8500 if P > 13 else 6400
    if op == W.M2L and P > 18:
        n = 25000 if P <= 20 else 33000
    parts += [physical_batch(orc, op, 1, P, n, 3 * P + op)]
    items, src, nd = join(parts)
    if op != W.M2L:
        for c in "xyz":
            items[c][5:60:7] = 0.0
    k = len(parts[0][0]) + 4 * (P - 1)
    items = np.concatenate([items[:k], np.random.default_rng(P).permutation(items[k:])])
    dst0 = 1e-3 * np.resize(src, nd)
    check(sfmm, orc, op, items, src, dst0, f"op {op} P={P} n={len(items)}")


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("P", [7, 10, 14, 16, 19])
def test_octet_runs(sfmm, orc, op, P):
    """Repeated targets: runs of 1 to 40 items that begin and end anywhere in
    a group, with zero shifts and other orders between them."""
    rng = np.random.default_rng(3 * P + op)
    n = 12800 if P > 18 else 8500
    if op == W.M2L and P > 18:
        n = 25000
    parts = [physical_batch(orc, op, P, P, 400, 7 * P + op)]
    if op != W.L2L:
        parts += [physical_batch(orc, op, P, 3, 40, 8 * P + op)]
    parts += [physical_batch(orc, op, 2, P, n, 9 * P + op)]
    blocks = []
    for it, s, d in parts:
        it = it.copy()
        pout = int(it["p_out"][0])
        target = np.repeat(np.arange(len(it)), rng.integers(1, 41, len(it)))[:len(it)]
        it["dst"] = target.astype(np.uint64) * np.uint64(pout * (pout + 1))
        blocks.append((it, s, d))
    items, src, nd = join(blocks)
    if op != W.M2L:
        for c in "xyz":
            items[c][3:400:11] = 0.0
    check(sfmm, orc, op, items, src, np.zeros(nd), f"runs op {op} P={P} n={len(items)}")


@pytest.mark.parametrize("P", [8, 9, 11, 12])
@pytest.mark.parametrize("n", [512, 513])
def test_small_m2l_default(sfmm, orc, P, n):
    """Both sides of the item count up to which M2L of orders 9 to 11 stays on
    lanes."""
    items, src, dst = physical_batch(orc, W.M2L, P, P, n, P + n)
    ctx = sfmm.Context(P)
    plan = sfmm.Plan(ctx, W.M2L, items)
    assert plan.launch_info()[0][0] == (1 if n == 512 and 9 <= P <= 11 else MFMA)
    d = torch.zeros(len(dst), dtype=torch.float64, device="cuda")
    plan.execute(torch.from_numpy(src).to("cuda"), d)
    torch.cuda.synchronize()
    want = orc.translate(W.M2L, items, src, np.zeros(len(dst)))
    naive = orc.translate(W.M2L, items, src, np.zeros(len(dst)), naive=True)
    tol = max(20 * block_errors(naive, want, np.zeros(len(dst)), items).max(), 1e-13)
    assert block_errors(d.cpu().numpy(), want, np.zeros(len(dst)), items).max() <= tol


def test_noalloc_long_runs(sfmm, orc):
    """Repeated targets whose blocks fit the fixed scratch array with runs of
    16 items, not of 8: M2L of order 16, 240,000 items (all but 200 of them
    of orders (1, 16)) in runs of 16."""
    import ctypes
    n, P = 240000, 16
    parts = [physical_batch(orc, W.M2L, P, P, 200, 1), physical_batch(orc, W.M2L, 1, P, n - 200, 2)]
    items, src, nd = join(parts)
    rep = 16 * 20
    items["dst"] = (np.arange(n) // rep).astype(np.uint64) * np.uint64(P * (P + 1))
    order = np.lexsort((np.arange(n), items["p_in"]))
    items = items[order]
    nd = (n // rep + 1) * P * (P + 1)
    ctx = sfmm.Context(P)
    s, d = torch.from_numpy(src).to("cuda"), torch.zeros(nd, dtype=torch.float64, device="cuda")
    items = np.ascontiguousarray(items, dtype=W.ITEM_DTYPE)
    rc = sfmm.load().sfmm_translate_noalloc(ctx.handle, W.M2L, items.ctypes.data, n, s.data_ptr(), s.numel(),
                                            d.data_ptr(), d.numel(),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    e = torch.zeros_like(d)
    sfmm.Plan(ctx, W.M2L, items).execute(s, e)
    torch.cuda.synchronize()
    # sums of 320 results of one operator in two groupings: 1e-12 of the block
    a, b = d.cpu().numpy().reshape(-1, P * (P + 1)), e.cpu().numpy().reshape(-1, P * (P + 1))
    assert (np.linalg.norm(a - b, axis=1) <= 1e-12 * np.linalg.norm(b, axis=1) + 0.0).all()
