"""Performance cases of the translation engine, its particle operators and the
far-field evaluation, through the package's public entry points.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call, on the GPU
    run(state)          one pass through the entry points; its outputs
    work(case)          bytes and flops one pass cannot do without
    exact(case, seed)   the outputs in 64 bits by plain torch, where that is
                        a closed formula

Kinds of case and the ranges `draw` spreads over:

    translate  one list of independent translations of one order: M2M, M2L
               or L2L, orders 2..24 (random coefficients) or 25..48 (the
               expansions of point charges), 64 to 1,000,000 items; FP64, or
               FP32 arithmetic for M2L
    mixed      independent translations of many order pairs in one list
    lists      M2L interaction lists of a uniform grid of cells: every cell
               receives up to 189 neighbours' expansions
    p2m, l2p   charges to multipoles, locals to potentials and gradients,
               1 or 3 charges per point, ragged cells
    fmm        the whole far-field evaluation of a Plummer sphere

Coefficients of an expansion of order P: Re C_n^m at n(n+1)+m and Im C_n^m
at (n+1)^2+m, degrees n < P, P(P+1) reals.
"""
import math

import numpy as np
import torch

import solidfmm_amd
from solidfmm_amd import CELL_DTYPE, ITEM_DTYPE, CellSet, Context, Plan
from solidfmm_amd.fmm import FMM

DEV = "cuda:0"
OPS = {"m2m": 0, "m2l": 1, "l2l": 2}
PRECISIONS = {"fp64": solidfmm_amd.SFMM_FP64, "fp32": solidfmm_amd.SFMM_FP32}

# Bytes no pass may move more of than the largest listed case (M2M of order
# 16 on a million items), and flops (the Plummer sphere's).
MOST_BYTES = 6.6e9
MOST_FLOPS = 3.0e10


def listed():
    return [
        # the M2M/L2L of a few cells of a small tree, or one request of a
        # serving loop: launch and latency bound
        {"name": "m2l_p8_n500", "kind": "translate", "op": "m2l", "p": 8, "n": 500, "precision": "fp64"},
        # the benchmark's headline: one batch of M2L translations
        {"name": "m2l_p10_n100000", "kind": "translate", "op": "m2l", "p": 10, "n": 100_000, "precision": "fp64"},
        # upward pass of a large tree at high accuracy, the largest batch
        {"name": "m2m_p16_n1000000", "kind": "translate", "op": "m2m", "p": 16, "n": 1_000_000, "precision": "fp64"},
        # downward pass, a ragged count and an odd order
        {"name": "l2l_p13_n77777", "kind": "translate", "op": "l2l", "p": 13, "n": 77_777, "precision": "fp64"},
        # M2L at the accuracy of the root's cells
        {"name": "m2l_p20_n30011", "kind": "translate", "op": "m2l", "p": 20, "n": 30_011, "precision": "fp64"},
        # beyond order 24: near machine precision, few cells
        {"name": "m2l_p32_n2003", "kind": "translate", "op": "m2l", "p": 32, "n": 2_003, "precision": "fp64"},
        # FP32 arithmetic on FP64 pools
        {"name": "m2l_fp32_p16_n200000", "kind": "translate", "op": "m2l", "p": 16, "n": 200_000,
         "precision": "fp32"},
        # an adaptive tree's lists: every order pair of 4..20 in one list
        {"name": "m2l_mixed_4_20_n500000", "kind": "mixed", "op": "m2l", "pmin": 4, "pmax": 20, "n": 500_000},
        # the M2L phase of one level of a uniform tree: targets repeat
        {"name": "m2l_lists_p8_side14", "kind": "lists", "p": 8, "side": 14},
        # leaves of a vortex method's tree (three charges per point)
        {"name": "p2m_p8_d3_250000", "kind": "p2m", "p": 8, "points": 250_000, "per_cell": 24, "dim": 3},
        # potentials and gradients of a gravity code's leaves
        {"name": "l2p_p10_d1_500000", "kind": "l2p", "p": 10, "points": 500_000, "per_cell": 32, "dim": 1},
        # P2M, M2M, M2L, L2L, L2P: orders 20 at the root to 6 at the leaves
        {"name": "fmm_plummer_100000", "kind": "fmm", "points": 100_000, "leaf": 64, "theta": 0.6, "p_root": 20,
         "p_leaf": 6},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["translate", "translate", "translate", "high", "fp32", "mixed", "lists", "p2m", "l2p",
                           "fmm"])
        if kind == "translate":
            case = {"kind": "translate", "op": rng.choice(["m2m", "m2l", "l2l"]), "p": rng.randint(2, 24),
                    "n": _log_int(rng, 64, 1_000_000), "precision": "fp64"}
        elif kind == "high":
            case = {"kind": "translate", "op": rng.choice(["m2m", "m2l", "l2l"]), "p": rng.randint(25, 48),
                    "n": _log_int(rng, 64, 4_000), "precision": "fp64"}
        elif kind == "fp32":
            case = {"kind": "translate", "op": "m2l", "p": rng.randint(4, 24), "n": _log_int(rng, 1_000, 300_000),
                    "precision": "fp32"}
        elif kind == "mixed":
            pmin = rng.randint(2, 10)
            case = {"kind": "mixed", "op": rng.choice(["m2m", "m2l", "l2l"]), "pmin": pmin,
                    "pmax": rng.randint(pmin + 2, 20), "n": _log_int(rng, 5_000, 500_000)}
        elif kind == "lists":
            case = {"kind": "lists", "p": rng.randint(3, 14), "side": rng.randint(5, 16)}
        elif kind in ("p2m", "l2p"):
            case = {"kind": kind, "p": rng.randint(3, 16), "points": _log_int(rng, 10_000, 1_000_000),
                    "per_cell": _log_int(rng, 8, 128), "dim": rng.choice([1, 3])}
        else:
            p_root = rng.randint(8, 20)
            case = {"kind": "fmm", "points": _log_int(rng, 20_000, 100_000), "leaf": rng.choice([32, 64, 100]),
                    "theta": rng.choice([0.5, 0.6, 0.7]), "p_root": p_root, "p_leaf": rng.randint(4, min(8, p_root))}
        w = work(case)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS:
            return case


# ---------------------------------------------------------------- sizes

def _size(p):
    return p * (p + 1)


def _flops(op, p):
    """Rotation scheme: 4 swaps of (n+1)^2 multiply-adds and 14 flops per
    coefficient of rotations on each side, and the z-translation's sums."""
    s2 = sum(k * k for k in range(1, p + 1))
    z = sum(4 * (p - m) ** 2 if op == "m2l" else 2 * (p - m) * (p - m + 1) for m in range(p))
    return 8 * s2 + 14 * p * (p + 1) + z


def _pair_count(side):
    """Directed M2L pairs of a side^3 grid: same-level cells whose parents
    (cells of the grid paired up) touch and which do not touch themselves."""
    total = near = 0
    for a in range(side):
        lo, hi = 2 * (a // 2 - 1), 2 * (a // 2 + 1) + 2
        total += min(hi, side) - max(lo, 0)
        near += min(a + 2, side) - max(a - 1, 0)
    return total ** 3 - near ** 3


def work(case):
    kind = case["kind"]
    if kind == "translate":
        n, p = case["n"], case["p"]
        return {"bytes": n * (24 * _size(p) + 24), "flops": n * _flops(case["op"], p)}
    if kind == "mixed":
        ps = range(case["pmin"], case["pmax"] + 1)
        size = sum(_size(p) for p in ps) / len(ps)
        flops = sum(_flops(case["op"], p) for p in ps) / len(ps)
        return {"bytes": int(case["n"] * (24 * size + 24)), "flops": int(case["n"] * flops)}
    if kind == "lists":
        cells, pairs = case["side"] ** 3, _pair_count(case["side"])
        return {"bytes": cells * 24 * _size(case["p"]) + 24 * pairs, "flops": pairs * _flops("m2l", case["p"])}
    if kind in ("p2m", "l2p"):
        n, p, d = case["points"], case["p"], case["dim"]
        cells = max(1, n // case["per_cell"])
        coef = p * (p + 1) // 2
        if kind == "p2m":
            return {"bytes": 8 * (n * (3 + d) + cells * d * 2 * _size(p)), "flops": n * coef * (8 + 4 * d)}
        return {"bytes": 8 * (n * (3 + d) + cells * d * _size(p) + 2 * 4 * d * n), "flops": n * coef * (8 + 16 * d)}
    # fmm: about 9 M2L pairs per point at theta 0.6, mostly at the leaves' order
    p = case["p_leaf"] + 2
    pairs = 9 * case["points"] * (0.6 / case["theta"]) ** 3 * 64 / case["leaf"]
    return {"bytes": int(case["points"] * 8 * (4 + 4 + 24 * _size(p) / 16)), "flops": int(pairs * _flops("m2l", p))}


# ---------------------------------------------------------------- harmonics

def _regular(p, x, y, z):
    """R_n^m (m >= 0) of degrees n < p at points x, y, z: {(n, m): complex}."""
    R = {(0, 0): torch.ones_like(x) + 0j}
    u = torch.complex(x, y)
    r2 = x * x + y * y + z * z
    for m in range(1, p):
        R[m, m] = R[m - 1, m - 1] * u / (2 * m)
    for m in range(p):
        if m + 1 < p:
            R[m + 1, m] = z * R[m, m]
        for n in range(m + 2, p):
            R[n, m] = ((2 * n - 1) * z * R[n - 1, m] - r2 * R[n - 2, m]) / ((n + m) * (n - m))
    return R


def _singular(p, x, y, z):
    """S_n^m (m >= 0) of degrees n < p: {(n, m): complex}."""
    r2 = x * x + y * y + z * z
    S = {(0, 0): 1 / torch.sqrt(r2) + 0j}
    u = torch.complex(x, y) / r2
    zz = z / r2
    for m in range(1, p):
        S[m, m] = (2 * m - 1) * u * S[m - 1, m - 1]
    for m in range(p):
        if m + 1 < p:
            S[m + 1, m] = (2 * m + 1) * zz * S[m, m]
        for n in range(m + 2, p):
            S[n, m] = (2 * n - 1) * zz * S[n - 1, m] - (n + m - 1) * (n - m - 1) / r2 * S[n - 2, m]
    return S


def _pack(H, p):
    """Harmonics as rows of P(P+1) reals in the expansion layout."""
    x = H[0, 0]
    out = torch.zeros((x.numel(), _size(p)), dtype=torch.float64, device=x.device)
    for n in range(p):
        for m in range(n + 1):
            out[:, n * (n + 1) + m] = H[n, m].real
            out[:, (n + 1) ** 2 + m] = H[n, m].imag
    return out


def _full(H, p):
    """Harmonics or coefficients of all orders -n..n as a tensor [items, p, 2p-1]
    (order m at column m + p - 1), by C_n^-m = (-1)^m conj(C_n^m)."""
    x = H[0, 0]
    out = torch.zeros((x.numel(), p, 2 * p - 1), dtype=torch.complex128, device=x.device)
    for n in range(p):
        for m in range(n + 1):
            out[:, n, p - 1 + m] = H[n, m]
            if m:
                out[:, n, p - 1 - m] = (-1) ** m * H[n, m].conj()
    return out


# ---------------------------------------------------------------- inputs

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000 + stream)
    return g


def _uniform(seed, stream, shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=_gen(seed, stream), dtype=torch.float64, device=DEV) * (hi - lo) + lo


def _directions(seed, stream, n):
    z = _uniform(seed, stream, n, -1.0, 1.0)
    phi = _uniform(seed, stream + 1, n, 0.0, 2 * math.pi)
    rho = torch.sqrt(torch.clamp(1 - z * z, min=0.0))
    return torch.stack([rho * torch.cos(phi), rho * torch.sin(phi), z], 1)


def _shifts(op, seed, n):
    """M2L: well-separated centres, |shift| in [2, 4]; M2M and L2L: from a
    cell's centre to that of one of its octants, or back."""
    if op == "m2l":
        return _directions(seed, 20, n) * _uniform(seed, 22, (n, 1), 2.0, 4.0)
    signs = torch.where(_uniform(seed, 23, (n, 3)) < 0.5, -1.0, 1.0).double()
    return 0.5 * signs * _uniform(seed, 24, (n, 1), 0.5, 1.0)


def _random_blocks(seed, stream, n, p):
    a = _uniform(seed, stream, (n, _size(p)), -1.0, 1.0)
    a[:, [(k + 1) ** 2 for k in range(p)]] = 0.0  # Im C_n^0
    return a


def _charge_blocks(op, seed, n, p):
    """Multipoles of a charge inside the cell (M2M, M2L), locals of one
    outside it (L2L): what orders beyond 24 meet in use."""
    q = _directions(seed, 30, n) * _uniform(seed, 32, (n, 1), 0.1, 0.8)
    if op == "l2l":
        q = _directions(seed, 33, n) * _uniform(seed, 35, (n, 1), 3.0, 4.5)
        return _pack(_singular(p, *q.unbind(1)), p)
    return _pack(_regular(p, *q.unbind(1)), p)


def _source_blocks(case, seed, n):
    if case["p"] > 24:
        return _charge_blocks(case["op"], seed, n, case["p"])
    return _random_blocks(seed, 1, n, case["p"])


def _items(src, dst, p_in, p_out, shifts):
    it = np.zeros(len(src), dtype=ITEM_DTYPE)
    it["src"], it["dst"], it["p_in"], it["p_out"] = src, dst, p_in, p_out
    sh = shifts.cpu().numpy()
    it["x"], it["y"], it["z"] = sh[:, 0], sh[:, 1], sh[:, 2]
    return it


def _mixed_orders(case, seed):
    """Every order of pmin..pmax equally often, in an order of the seed's."""
    rng = np.random.default_rng(seed)
    orders = case["pmin"] + np.arange(case["n"]) % (case["pmax"] - case["pmin"] + 1)
    return rng.permutation(orders), rng.permutation(orders)


def _mixed_pool(case, seed, p_in, offsets):
    src = _uniform(seed, 1, int(_size(p_in).sum()), -1.0, 1.0)
    for n in range(case["pmax"]):  # Im C_n^0
        src[torch.from_numpy(offsets[p_in > n] + (n + 1) ** 2).to(DEV)] = 0.0
    return src


def _offsets(sizes):
    return np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)


def _grid_pairs(side):
    """(source, target) cells of the grid's interaction lists, by target."""
    a = np.arange(side)
    near = np.abs(a[:, None] - a[None, :]) <= 1
    par = np.abs(a[:, None] // 2 - a[None, :] // 2) <= 1
    t, s = np.nonzero(par)  # per axis: candidate source of each target
    k = len(t)
    i, j, l = (v.ravel() for v in np.meshgrid(np.arange(k), np.arange(k), np.arange(k), indexing="ij"))
    touch = near[t[i], s[i]] & near[t[j], s[j]] & near[t[l], s[l]]
    i, j, l = i[~touch], j[~touch], l[~touch]
    tgt = (t[i] * side + t[j]) * side + t[l]
    src = (s[i] * side + s[j]) * side + s[l]
    order = np.argsort(tgt, kind="stable")
    return src[order], tgt[order]


def _cells(case, seed):
    """Ragged cells (1 to about twice the mean, in an order of the seed's)
    over all points: (first, count, centre), and the points (x, y, z,
    charges) on the GPU."""
    n, mean, d = case["points"], case["per_cell"], case["dim"]
    rng = np.random.default_rng(seed)
    count = 1 + np.arange(2 * n // mean + 2 * mean) % (2 * mean - 1)
    count = count[: int(np.searchsorted(np.cumsum(count), n)) + 1]
    count[-1] -= int(count.sum()) - n
    count = rng.permutation(count)
    first = _offsets(count)
    centre = rng.uniform(-10.0, 10.0, (len(count), 3))
    cell_of = torch.from_numpy(np.repeat(np.arange(len(count)), count)).to(DEV)
    pts = torch.empty((n, 3 + d), dtype=torch.float64, device=DEV)
    pts[:, :3] = torch.from_numpy(centre).to(DEV)[cell_of] + _uniform(seed, 40, (n, 3), -0.5, 0.5)
    pts[:, 3:] = _uniform(seed, 41, (n, d), -1.0, 1.0)
    return first, count, centre, cell_of, pts


def _local_blocks(case, seed, blocks):
    """Local expansions of a charge well outside the cell."""
    p = case["p"]
    q = _directions(seed, 50, blocks) * _uniform(seed, 52, (blocks, 1), 2.0, 4.0)
    return _pack(_singular(p, *q.unbind(1)), p)


def _plummer(case, seed):
    """Plummer sphere of scale radius 1 (r = 1/sqrt(u^(-2/3) - 1), isotropic),
    with charges."""
    n = case["points"]
    rng = np.random.default_rng(seed)
    r = np.minimum(1 / np.sqrt(rng.uniform(1e-12, 1.0, n) ** (-2 / 3) - 1 + 1e-15), 100.0)
    z = rng.uniform(-1, 1, n)
    phi = rng.uniform(0, 2 * math.pi, n)
    s = np.sqrt(1 - z * z)
    return np.stack([r * s * np.cos(phi), r * s * np.sin(phi), r * z, rng.uniform(0.5, 1.5, n) / n], 1)


# ---------------------------------------------------------------- passes

def prepare(case, seed):
    solidfmm_amd.load()
    kind = case["kind"]
    if kind == "translate":
        n, p = case["n"], case["p"]
        ctx = Context(p, precision=PRECISIONS[case["precision"]])
        off = np.arange(n) * _size(p)
        items = _items(off, off, p, p, _shifts(case["op"], seed, n))
        return {"do": "plan", "ctx": ctx, "plan": Plan(ctx, OPS[case["op"]], items),
                "src": _source_blocks(case, seed, n).reshape(-1),
                "dst": torch.zeros(n * _size(p), dtype=torch.float64, device=DEV)}
    if kind == "mixed":
        p_in, p_out = _mixed_orders(case, seed)
        so, do = _offsets(_size(p_in)), _offsets(_size(p_out))
        src = _mixed_pool(case, seed, p_in, so)
        ctx = Context(case["pmax"])
        items = _items(so, do, p_in, p_out, _shifts(case["op"], seed, case["n"]))
        return {"do": "plan", "ctx": ctx, "plan": Plan(ctx, OPS[case["op"]], items), "src": src,
                "dst": torch.zeros(int(_size(p_out).sum()), dtype=torch.float64, device=DEV)}
    if kind == "lists":
        p, side = case["p"], case["side"]
        s, t = _grid_pairs(side)
        ctr = _grid_centres(side)
        ctx = Context(p)
        items = _items(s * _size(p), t * _size(p), p, p, ctr[t] - ctr[s])
        q = _directions(seed, 60, side ** 3) * _uniform(seed, 62, (side ** 3, 1), 0.05, 0.45)
        src = _pack(_regular(p, *q.unbind(1)), p).reshape(-1)
        return {"do": "plan", "ctx": ctx, "plan": Plan(ctx, OPS["m2l"], items), "src": src,
                "dst": torch.zeros(side ** 3 * _size(p), dtype=torch.float64, device=DEV)}
    if kind in ("p2m", "l2p"):
        p, d = case["p"], case["dim"]
        first, count, centre, _, pts = _cells(case, seed)
        cells = np.zeros(len(count), dtype=CELL_DTYPE)
        cells["x"], cells["y"], cells["z"] = centre.T
        cells["offset"] = np.arange(len(count)) * d * _size(p)
        cells["first"], cells["count"], cells["order"], cells["dim"] = first, count, p, d
        ctx = Context(p)
        state = {"do": kind, "ctx": ctx, "cells": CellSet(ctx, cells, case["points"]), "points": pts}
        if kind == "p2m":
            state["pool"] = torch.zeros(len(count) * d * _size(p), dtype=torch.float64, device=DEV)
        else:
            state["pool"] = _local_blocks(case, seed, len(count) * d).reshape(-1)
            state["phi"] = torch.zeros((case["points"], d), dtype=torch.float64, device=DEV)
            state["grad"] = torch.zeros((case["points"], d, 3), dtype=torch.float64, device=DEV)
        return state
    ctx = Context(case["p_root"])
    fmm = FMM(ctx, _plummer(case, seed), leaf_size=case["leaf"], theta=case["theta"], p_root=case["p_root"],
              p_leaf=case["p_leaf"])
    return {"do": "fmm", "ctx": ctx, "fmm": fmm}


def _grid_centres(side):
    """Centres of the grid's unit cells, a little off the middle as smallest
    balls' centres are."""
    g = torch.arange(side ** 3, device=DEV)
    c = torch.stack([g // (side * side), g // side % side, g % side], 1).double()
    return c + 0.1 * torch.sin(torch.arange(3 * side ** 3, device=DEV).double()).reshape(-1, 3)


def run(state):
    do = state["do"]
    if do == "plan":
        state["plan"].execute(state["src"], state["dst"])
        return state["dst"]
    if do == "p2m":
        state["cells"].p2m(state["points"], state["pool"])
        return state["pool"]
    if do == "l2p":
        state["cells"].l2p(state["points"], state["pool"], state["phi"], state["grad"])
        return {"phi": state["phi"], "grad": state["grad"]}
    phi, grad = state["fmm"].evaluate()
    return {"phi": phi, "grad": grad}


# ---------------------------------------------------------------- 64 bits

def _naive(op, blocks, shifts, p_in, p_out):
    """The operators' defining sums for items of one order pair: [items, P_out(P_out+1)].

    M2M  M'_n^m = sum_{k,l} M_k^l R_{n-k}^{m-l}(-shift)
    M2L  L_n^m  = (-1)^n sum_{k,l} conj(M_k^l) S_{n+k}^{m+l}(shift)
    L2L  L'_n^m = sum_{k,l} L_k^l conj(R_{k-n}^{l-m}(shift))
    """
    out = torch.empty((len(blocks), _size(p_out)), dtype=torch.float64, device=DEV)
    ph = p_in + p_out
    step = max(1, int(6e8 // (16 * ph * (2 * ph - 1) * 2)))
    for a in range(0, len(blocks), step):
        b, sh = blocks[a:a + step], shifts[a:a + step]
        x, y, z = sh.unbind(1)
        C = _full({(n, m): torch.complex(b[:, n * (n + 1) + m], b[:, (n + 1) ** 2 + m])
                   for n in range(p_in) for m in range(n + 1)}, p_in)
        if op == "m2l":
            H = _full(_singular(ph, x, y, z), ph)
        elif op == "m2m":
            H = _full(_regular(ph, -x, -y, -z), ph)
        else:
            H = _full(_regular(ph, x, y, z), ph).conj().resolve_conj()
        L = torch.zeros((len(b), p_out, p_out), dtype=torch.complex128, device=DEV)
        for k in range(p_in):
            for l in range(-k, k + 1):
                c = C[:, k, p_in - 1 + l, None, None]
                # columns of orders m + l, m - l or l - m for m = 0..p_out-1
                if op == "m2l":
                    L += c.conj() * H[:, k:k + p_out, ph - 1 + l:ph - 1 + l + p_out]
                elif op == "m2m" and k < p_out:
                    L[:, k:] += c * H[:, :p_out - k, ph - 1 - l:ph - 1 - l + p_out]
                elif op == "l2l":
                    e = min(k + 1, p_out)  # degrees n <= k, from H's degrees k - n
                    L[:, :e] += c * H[:, k - e + 1:k + 1, ph - 1 + l - p_out + 1:ph + l].flip(1, 2)
        for n in range(p_out):
            s = -1.0 if op == "m2l" and n & 1 else 1.0
            out[a:a + step, n * (n + 1):n * (n + 1) + n + 1] = s * L[:, n, :n + 1].real
            out[a:a + step, (n + 1) ** 2:(n + 1) ** 2 + n + 1] = s * L[:, n, :n + 1].imag
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "translate":
        n, p = case["n"], case["p"]
        if n * p ** 4 > 7e10:
            return None
        return _naive(case["op"], _source_blocks(case, seed, n), _shifts(case["op"], seed, n), p, p).reshape(-1)
    if kind == "mixed":
        if case["n"] * case["pmax"] ** 4 > 1e11:
            return None
        p_in, p_out = _mixed_orders(case, seed)
        so, do = _offsets(_size(p_in)), _offsets(_size(p_out))
        src, shifts = _mixed_pool(case, seed, p_in, so), _shifts(case["op"], seed, case["n"])
        out = torch.empty(int(_size(p_out).sum()), dtype=torch.float64, device=DEV)
        for a, b in sorted(set(zip(p_in.tolist(), p_out.tolist()))):
            sel = np.nonzero((p_in == a) & (p_out == b))[0]
            i = torch.from_numpy(so[sel]).to(DEV)[:, None] + torch.arange(_size(a), device=DEV)
            j = torch.from_numpy(do[sel]).to(DEV)[:, None] + torch.arange(_size(b), device=DEV)
            out[j] = _naive(case["op"], src[i], shifts[torch.from_numpy(sel).to(DEV)], a, b)
        return out
    if kind == "lists":
        p, side = case["p"], case["side"]
        if _pair_count(side) * p ** 4 > 2e10:
            return None
        s, t = _grid_pairs(side)
        ctr = _grid_centres(side)
        q = _directions(seed, 60, side ** 3) * _uniform(seed, 62, (side ** 3, 1), 0.05, 0.45)
        src = _pack(_regular(p, *q.unbind(1)), p)
        s, t = torch.from_numpy(s).to(DEV), torch.from_numpy(t).to(DEV)
        out = torch.zeros((side ** 3, _size(p)), dtype=torch.float64, device=DEV)
        out.index_add_(0, t, _naive("m2l", src[s], ctr[t] - ctr[s], p, p))
        return out.reshape(-1)
    if kind == "p2m":
        p, d = case["p"], case["dim"]
        _, count, centre, cell_of, pts = _cells(case, seed)
        R = _regular(p, *(pts[:, :3] - torch.from_numpy(centre).to(DEV)[cell_of]).unbind(1))
        out = torch.zeros((len(count), d, _size(p)), dtype=torch.float64, device=DEV)
        for (n, m), h in R.items():
            for part, at in ((h.real, n * (n + 1) + m), (h.imag, (n + 1) ** 2 + m)):
                v = torch.zeros((len(count), d), dtype=torch.float64, device=DEV)
                out[:, :, at] = v.index_add_(0, cell_of, part[:, None] * pts[:, 3:])
        return out.reshape(-1)
    if kind == "l2p":
        p, d = case["p"], case["dim"]
        _, count, centre, cell_of, pts = _cells(case, seed)
        R = _regular(p, *(pts[:, :3] - torch.from_numpy(centre).to(DEV)[cell_of]).unbind(1))
        L = _local_blocks(case, seed, len(count) * d).reshape(len(count), d, -1)
        phi = torch.zeros((case["points"], d), dtype=torch.float64, device=DEV)
        grad = torch.zeros((case["points"], d, 3), dtype=torch.float64, device=DEV)

        def lower(n, m):  # R_{n-1}^m of any order m
            if n == 0 or abs(m) > n - 1:
                return torch.zeros_like(R[0, 0])
            return R[n - 1, m] if m >= 0 else (-1) ** m * R[n - 1, -m].conj()

        for (n, m), h in R.items():
            w = 2.0 if m else 1.0
            c = torch.complex(L[:, :, n * (n + 1) + m], -L[:, :, (n + 1) ** 2 + m])[cell_of]
            dx = (lower(n, m - 1) - lower(n, m + 1)) / 2
            dy = (lower(n, m - 1) + lower(n, m + 1)) * 0.5j
            phi += w * (c * h[:, None]).real
            for k, g in enumerate((dx, dy, lower(n, m))):
                grad[:, :, k] += w * (c * g[:, None]).real
        return {"phi": phi, "grad": grad}
    return None  # fmm: truncated expansions of thousands of cells
