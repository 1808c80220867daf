"""P2M and L2P over sets of so many cells that a wave takes several -- needs
an MI355X.  Cells of 0 to 70 points (several in one chunk of 64 lanes, and
chunks within a cell) against plain FP64 sums over the oracle's harmonics on a
sample of cells; tolerances as in test_gpu_particles.py (1e-13 for sums of R,
1e-12 for dot products with random coefficients)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def sfmm():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    import solidfmm_amd
    solidfmm_amd.load()
    return solidfmm_amd


def make(sfmm, n_cells, orders, D, seed):
    rng = np.random.default_rng(seed)
    counts = rng.integers(0, 9, n_cells)
    counts[::7] = rng.integers(30, 71, len(counts[::7]))
    P = rng.choice(orders, n_cells)
    cells = np.zeros(n_cells, dtype=sfmm.CELL_DTYPE)
    ctr = rng.uniform(-2, 2, (n_cells, 3))
    cells["x"], cells["y"], cells["z"] = ctr.T
    size = D * P * (P + 1) + 2
    cells["offset"] = np.cumsum(size) - size
    cells["first"] = np.cumsum(counts) - counts
    cells["count"], cells["order"], cells["dim"] = counts, P, D
    pts = np.concatenate([np.repeat(ctr, counts, axis=0) + rng.uniform(-0.5, 0.5, (counts.sum(), 3)),
                          rng.uniform(-1, 1, (counts.sum(), D))], axis=1)
    sample = np.concatenate([np.arange(24), rng.choice(n_cells, 40, replace=False), [n_cells - 2, n_cells - 1]])
    return cells, pts, int(size.sum()), sample


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


# 2: L2P without a walk; 16, 3: several staged blocks a wave do not all fit
@pytest.mark.parametrize("n_cells,orders,D", [(6000, [8], 1), (15000, [3, 4, 7], 1), (12000, [9], 3),
                                              (24000, [16, 3], 4), (7000, [2], 2), (5800, [33, 5], 1)])
def test_runs_of_cells(sfmm, n_cells, orders, D):
    orc = oracle.Oracle()
    cells, pts, plen, sample = make(sfmm, n_cells, orders, D, n_cells + D)
    rng = np.random.default_rng(5)
    pool0 = rng.standard_normal(plen)
    cs = sfmm.CellSet(sfmm.Context(max(orders)), cells, len(pts))
    pool, phi, grad = dev(pool0), dev(np.zeros((len(pts), D))), dev(np.zeros((len(pts), D, 3)))
    cs.l2p(dev(pts), pool, phi, grad)
    cs.p2m(dev(pts), pool)
    torch.cuda.synchronize()
    got, phi, grad = pool.cpu().numpy(), phi.cpu().numpy(), grad.cpu().numpy()
    untouched = np.ones(plen, bool)
    for c in cells:
        P = int(c["order"])
        untouched[int(c["offset"]):int(c["offset"]) + D * P * (P + 1)] = False
    assert np.array_equal(got[untouched], pool0[untouched])
    for s in sample:
        c = cells[s]
        P, o, first, n = int(c["order"]), int(c["offset"]), int(c["first"]), int(c["count"])
        B = P * (P + 1)
        blocks = pool0[o:o + D * B].reshape(D, B)
        want = blocks.copy()
        ph, gr = np.zeros((n, D)), np.zeros((n, D, 3))
        for i in range(n):
            d = pts[first + i, :3] - np.array([c["x"], c["y"], c["z"]])
            R = orc.harmonic("R", P, *d)
            dR = orc.harmonic("dR", P, *d).reshape(3, -1)
            for k in range(D):
                want[k] += pts[first + i, 3 + k] * R
                b = np.ascontiguousarray(blocks[k])
                ph[i, k] = orc.dot(b, P, R, P)
                gr[i, k] = [orc.dot(b, P, np.ascontiguousarray(g), P) for g in dR]
        assert np.abs(got[o:o + D * B] - want.reshape(-1)).max() <= 1e-13 * max(np.abs(want).max(), 1), (s, P, n)
        if n:
            assert np.abs(phi[first:first + n] - ph).max() <= 1e-12 * np.abs(ph).max(), (s, P, n)
            assert np.abs(grad[first:first + n] - gr).max() <= 1e-12 * max(np.abs(gr).max(), 1e-300), (s, P, n)


# Both sides of the lines between a wave per cell and runs of cells: points a
# cell (4 and 5 at 512 cells, 6 and 7 above, 3 and 4 or 4 and 5 of higher
# orders), a larger cell among them (24 and 25 points of 6 a cell on average),
# 5120 and 5121 cells of order 4, the share of lanes with a point (26 and 27 of
# 64), the cells (767 and 768), a cell of two chunks, the orders' ends; and
# cells of two orders, every fourth of the first.
@pytest.mark.parametrize("n_cells,count,largest,orders,D", [
    (512, 4, 4, [8], 1), (512, 5, 5, [8], 1), (513, 6, 6, [10], 2), (513, 7, 7, [10], 2), (600, 5, 24, [6], 1),
    (600, 5, 25, [6], 1), (1024, 3, 3, [12], 2), (1024, 4, 4, [12], 2), (1100, 4, 4, [16], 3), (1100, 5, 5, [16], 3),
    (1100, 3, 3, [32], 1), (17000, 2, 2, [8], 3), (17000, 1, 1, [1], 2), (5120, 9, 9, [4], 2), (5121, 9, 9, [4], 2),
    (768, 27, 27, [8], 4), (768, 26, 26, [8], 4), (767, 27, 27, [8], 4), (1000, 64, 65, [8], 4), (3100, 40, 40, [5], 1),
    (2000, 2, 2, [16, 5], 1), (2000, 3, 3, [16, 5], 1), (3100, 20, 20, [10, 3], 3), (6000, 8, 8, [10, 3], 3),
    (3100, 64, 65, [24, 8], 4)])
def test_sides_of_the_lines(sfmm, n_cells, count, largest, orders, D):
    orc = oracle.Oracle()
    rng = np.random.default_rng(n_cells + 10 * count + orders[0])
    order = np.where(np.arange(n_cells) % 4 == 0, orders[0], orders[-1])
    counts = np.full(n_cells, count)
    counts[n_cells // 2] = largest
    cells = np.zeros(n_cells, dtype=sfmm.CELL_DTYPE)
    ctr = rng.uniform(-2, 2, (n_cells, 3))
    cells["x"], cells["y"], cells["z"] = ctr.T
    size = D * order * (order + 1)
    cells["offset"] = np.cumsum(size) - size
    cells["first"] = np.cumsum(counts) - counts
    cells["count"], cells["order"], cells["dim"] = counts, order, D
    n = int(counts.sum())
    pts = np.concatenate([np.repeat(ctr, counts, axis=0) + rng.uniform(-0.5, 0.5, (n, 3)),
                          rng.uniform(-1, 1, (n, D))], axis=1)
    pool0 = rng.standard_normal(int(size.sum()))
    cs = sfmm.CellSet(sfmm.Context(max(orders)), cells, n)
    pool, phi, grad = dev(pool0), dev(np.zeros((n, D))), dev(np.zeros((n, D, 3)))
    cs.l2p(dev(pts), pool, phi, grad)
    cs.p2m(dev(pts), pool)
    torch.cuda.synchronize()
    got, phi, grad = pool.cpu().numpy(), phi.cpu().numpy(), grad.cpu().numpy()
    for s in [0, 1, 7, n_cells // 2, n_cells - 2, n_cells - 1]:
        P = int(order[s])
        block = slice(int(cells["offset"][s]), int(cells["offset"][s] + size[s]))
        blocks = pool0[block].reshape(D, -1)
        want = blocks.copy()
        at = slice(int(cells["first"][s]), int(cells["first"][s]) + int(counts[s]))
        ph, gr = np.zeros((counts[s], D)), np.zeros((counts[s], D, 3))
        for i, p in enumerate(pts[at]):
            d = p[:3] - ctr[s]
            R, dR = orc.harmonic("R", P, *d), orc.harmonic("dR", P, *d).reshape(3, -1)
            for k in range(D):
                want[k] += p[3 + k] * R
                b = np.ascontiguousarray(blocks[k])
                ph[i, k] = orc.dot(b, P, R, P)
                gr[i, k] = [orc.dot(b, P, np.ascontiguousarray(g), P) for g in dR]
        assert np.abs(got[block] - want.reshape(-1)).max() <= 1e-13 * max(np.abs(want).max(), 1), s
        assert np.abs(phi[at] - ph).max() <= 1e-12 * np.abs(ph).max(), s
        assert np.abs(grad[at] - gr).max() <= 1e-12 * max(np.abs(gr).max(), 1e-300), s
