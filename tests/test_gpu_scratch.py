"""Scratch memory of plans of repeated targets: what fits with the longest
runs runs -- needs an MI355X."""
import ctypes

import numpy as np
import pytest

from solidfmm_amd import serving as S
from solidfmm_amd import workload as W
from tests.test_gpu_lane_runs import repeated
from tests.test_gpu_octet import join
from tests.test_gpu_team import block_errors, sfmm  # noqa: F401
from tests.test_gpu_translate import physical_batch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LANE, MFMA = 1, 2
ARRAY = 64 << 20  # SFMM_NOALLOC_SCRATCH_BYTES


def within(sfmm, ctx, op, items, max_bytes):
    """A plan for an arena of max_bytes, bound to one."""
    plan = sfmm.Plan(ctx, op, items, prepared=True, max_bytes=max_bytes)
    arena = torch.empty(plan.device_bytes + 256, dtype=torch.uint8, device="cuda")
    off = -arena.data_ptr() % 256
    plan.bind(arena.data_ptr() + off, plan.device_bytes)
    return plan, arena


# Runs that begin and end anywhere in a pair of octet groups, with zero shifts
# and other orders between them, in lists whose last pair is one group: the
# orders with kernels for pairs, and one on either side (team kernels)
@pytest.mark.parametrize("op", [W.M2M, W.M2L, W.L2L])
@pytest.mark.parametrize("P", [12, 13, 14, 15, 16, 17, 18])
def test_longer_runs(sfmm, orc, op, P):
    parts = [repeated(orc, op, P, P, 300, [1, 16, 5, 40, 2, 9, 24], 7 * P + op),
             repeated(orc, op, 1, P, 33000 + 5, [16, 3, 17, 1, 8, 30], 9 * P + op)]
    if op != W.L2L:
        parts.insert(1, repeated(orc, op, P, 3, 40, [7, 16], 8 * P + op))
    items, src, nd = join(parts)
    if op != W.M2L:
        for c in "xyz":
            items[c][3:300:11] = 0.0
    ctx = sfmm.Context(P)
    ctx.set_kernels(MFMA)
    most = sfmm.Plan(ctx, op, items, prepared=True).device_bytes
    plan, arena = within(sfmm, ctx, op, items, most - 1)
    assert plan.device_bytes < most
    d = torch.zeros(nd, dtype=torch.float64, device="cuda")
    plan.execute(torch.from_numpy(src).to("cuda"), d)
    torch.cuda.synchronize()
    zero = np.zeros(nd)
    want = orc.translate(op, items, src, zero.copy())
    few = items[:200]
    few = few[np.unique(few["dst"], return_index=True)[1]]
    naive = block_errors(orc.translate(op, few, src, zero.copy(), naive=True),
                         orc.translate(op, few, src, zero.copy()), zero, few)
    tol = max(20 * naive.max(), 1e-13)
    err = block_errors(d.cpu().numpy(), want, zero, items).max()
    print(f"op {op} P={P}: {err:.2e} (tol {tol:.2e})", flush=True)
    assert err <= tol


# Lists that fit the array with longer runs than the faster kernels have: octets
# in pairs, a team, and lanes
@pytest.mark.parametrize("P,n,length,family", [(16, 240000, 16, MFMA), (13, 330000, 16, MFMA), (18, 200000, 24, MFMA),
                                                (10, 430000, 12, LANE)])
def test_noalloc_equals_plan(sfmm, orc, P, n, length, family):
    items, src, _ = physical_batch(orc, W.M2L, 1, P, n, P)
    items["dst"] = (np.arange(n) // length).astype(np.uint64) * np.uint64(P * (P + 1))
    nd = (n // length + 1) * P * (P + 1)
    items = np.ascontiguousarray(items, dtype=W.ITEM_DTYPE)
    ctx = sfmm.Context(P)
    plan = sfmm.Plan(ctx, W.M2L, items)
    assert plan.device_bytes <= ARRAY
    assert [i[0] for i in plan.launch_info()] == [family]
    s, d = torch.from_numpy(src).to("cuda"), torch.zeros(nd, dtype=torch.float64, device="cuda")
    e = torch.zeros_like(d)
    rc = sfmm.load().sfmm_translate_noalloc(ctx.handle, W.M2L, items.ctypes.data, n, s.data_ptr(), s.numel(),
                                            d.data_ptr(), d.numel(),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    plan.execute(s, e)
    torch.cuda.synchronize()
    assert torch.equal(d, e) and bool((d != 0).any())


def arena_case(orc):
    """20,000 M2L of order 10 into targets of 64 items, and an arena that
    holds their plan with runs of 64 only."""
    n, P = 20000, 10
    items, src, _ = physical_batch(orc, W.M2L, 1, P, n, 4)
    items["dst"] = (np.arange(n) // 64).astype(np.uint64) * np.uint64(P * (P + 1))
    blocks = n // 64 + 1
    budget = n * 48 + blocks * (8 * P * (P + 1) + 16 + 32) + 4096
    return items, src, blocks * P * (P + 1), P, (budget + 255) // 256 * 256


def test_prepare_within(sfmm, orc):
    items, src, nd, P, budget = arena_case(orc)
    ctx = sfmm.Context(P)
    plan = sfmm.Plan(ctx, W.M2L, items, prepared=True)
    assert plan.device_bytes > budget
    same = sfmm.Plan(ctx, W.M2L, items, prepared=True, max_bytes=plan.device_bytes)
    assert same.device_bytes == plan.device_bytes
    assert sfmm.Plan(ctx, W.M2L, items, prepared=True, max_bytes=budget).device_bytes <= budget


@pytest.mark.parametrize("kind", ["python", "native"])
def test_server_takes_what_fits(sfmm, orc, kind):
    items, src, nd, P, budget = arena_case(orc)
    ctx = sfmm.Context(P)
    pools = (torch.from_numpy(src).to("cuda"), torch.zeros(nd, dtype=torch.float64, device="cuda"))
    server = (S.Server if kind == "python" else S.NativeServer)(ctx, pools, 2, slots=1, budget_bytes=budget)
    request = S.Request(0, W.M2L, items, np.array([0]), np.array([1]))
    if kind == "python":
        server.run([request], realtime=False)
    else:
        rid = server.submit(request)
        assert server._lib.sfmm_server_drain(server._h) == 0
        rc, times = ctypes.c_int(), np.zeros(5)
        assert server._lib.sfmm_server_request_info(server._h, rid, times.ctypes.data, ctypes.byref(rc)) == 0
        assert rc.value == 0
        server.close()
    torch.cuda.synchronize()
    got = pools[1].cpu().numpy().reshape(-1, P * (P + 1))
    want = orc.translate(W.M2L, items, src, np.zeros(nd)).reshape(-1, P * (P + 1))
    # sums of 64 results of one operator in two groupings: 1e-12 of the block
    norm = np.linalg.norm(want, axis=1)
    assert (np.linalg.norm(got - want, axis=1) <= 1e-12 * norm).all() and (norm[:-1] > 0).all()
