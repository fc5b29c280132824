"""Performance cases: what a program does with the engine, from one small
product to the scale 22 sweep, each through an entry point of the C ABI
(include/gbo.h) or of its Python mirrors (gbo, gbo_torch).

Graphs are made on the GPU from the seed, as symmetric CSR without
self-loops or duplicates:

  rmat  power-law, quadrants .57/.19/.19/.05, edge factor `deg`, drawn at the
        next power of two and cut to n vertices (web and social graphs)
  er    G(n, m) with mean degree `deg` (evenly spread columns)
  king  8-neighbour grid, row-major numbering (meshes and road-like graphs:
        dense tiles near the diagonal, long shortest paths)

A state holds what such a program keeps: the packed matrix with its plan,
inputs, and output buffers where the entry point writes into the caller's.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "graph-bit-ops_amd"))

import gbo  # noqa: E402  (after torch: one HIP runtime for both)
import gbo_torch  # noqa: E402

DEV = "cuda"
RMAT = (0.57, 0.19, 0.19, 0.05)
WORD = {8: torch.uint8, 16: torch.int16, 32: torch.int32, 64: torch.int64}
INF = 0xFFFFFFFF
ALPHA = 0.85
PR_TOL = 1e-6   # L1 change that ends PageRank
PPR_TOL = 1e-6  # relative L1 change that ends both personalized solves
PPR_MAX = 200
MAX_LEVELS = 4096
SEEDS = 1000    # seed vertices of one personalization vector


def listed():
    return [
        # one product on a graph of a thousand vertices, the smallest call: what a caller that
        # multiplies many small graphs pays per call
        {"name": "count_er1k_bs32", "op": "count", "graph": "er", "n": 1024, "deg": 20, "bs": 32},
        # the headline sweep: y = A x over R-MAT scale 22 at the block size that is fastest for it
        {"name": "count_rmat22_bs8", "op": "count", "graph": "rmat", "n": 1 << 22, "deg": 16, "bs": 8},
        # pull BFS of a social graph: few levels, most of the work in two of them
        {"name": "bfs_rmat20_bs32", "op": "bfs", "graph": "rmat", "n": 1 << 20, "deg": 16, "bs": 32},
        # direction-optimizing BFS of a mesh: hundreds of levels with small frontiers
        {"name": "bfs_do_king512_bs8", "op": "bfs_do", "graph": "king", "n": 512 * 512, "deg": 8, "bs": 8},
        # weighted shortest paths, a vertex count that no block size divides
        {"name": "sssp_rmat_500k_bs16", "op": "sssp", "graph": "rmat", "n": 500_009, "deg": 16, "bs": 16},
        # PageRank of an ordinary evenly spread graph to a tolerance
        {"name": "pagerank_er200k_bs8", "op": "pagerank", "graph": "er", "n": 200_003, "deg": 16, "bs": 8},
        # connected components at the widest tile
        {"name": "cc_rmat20_bs64", "op": "cc", "graph": "rmat", "n": 1 << 20, "deg": 16, "bs": 64},
        # packing a CSR that is on the GPU: every new graph pays this once
        {"name": "pack_rmat20_bs64", "op": "pack", "graph": "rmat", "n": 1 << 20, "deg": 16, "bs": 64},
        # triangle counting by the masked product
        {"name": "tc_rmat18_bs32", "op": "tc", "graph": "rmat", "n": 1 << 18, "deg": 16, "bs": 32},
        # the general product C = L L^T with its integer values, on a mesh
        {"name": "spgemm_king1000_bs32", "op": "spgemm", "graph": "king", "n": 1000 * 1000, "deg": 8, "bs": 32},
        # 256 BFS runs in one pass (all-pairs samples, betweenness-like work)
        {"name": "msbfs_rmat18_256_bs8", "op": "msbfs", "graph": "rmat", "n": 1 << 18, "deg": 16, "bs": 8, "k": 256},
        # a training step through personalized PageRank: forward solve, then the gradients of the
        # teleport vectors and of alpha
        {"name": "ppr_rmat17_64_bs8", "op": "ppr", "graph": "rmat", "n": 1 << 17, "deg": 16, "bs": 8, "k": 64},
    ]


# op -> (smallest n, largest n, largest k)
RANGES = {
    "count": (1000, 1 << 22, 1), "sum": (1000, 1 << 22, 1), "min": (1000, 1 << 22, 1),
    "minplus": (1000, 1 << 22, 1), "bfs": (1000, 1 << 20, 1), "bfs_do": (1000, 1 << 20, 1),
    "sssp": (1000, 1 << 20, 1), "pagerank": (1000, 1 << 20, 1), "cc": (1000, 1 << 20, 1),
    "pack": (1000, 1 << 20, 1), "tc": (1000, 1 << 18, 1), "spgemm": (1000, 1_000_000, 1),
    "msbfs": (1000, 1 << 18, 256), "ppr": (1000, 1 << 17, 64),
}


def draw(rng):
    op = rng.choice(sorted(RANGES))
    lo, hi, kmax = RANGES[op]
    bs = rng.choice([8, 16, 32] if op == "ppr" else [8, 16, 32, 64])
    graph = rng.choice(["rmat", "rmat", "er", "king"])
    deg = rng.choice([8, 12, 16])
    if bs >= 32:  # a wide tile holds few nonzeros: the same memory at a quarter of the vertices
        hi = min(hi, 1 << 20)
    if op == "ppr":  # the wider tiles cost more a nonzero
        hi = hi * 8 // bs
    if graph == "king":
        deg = 8
        if op not in ("spgemm", "pack"):  # a level or an iteration per grid row
            hi = min(hi, 128 * 128 if op == "msbfs" else 512 * 512)
    elif op == "spgemm":  # L L^T grows with the square of the degree
        hi, deg, graph = 1 << 17, 4, "er"
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if graph == "king":
        n = int(math.isqrt(n)) ** 2
    case = {"op": op, "graph": graph, "n": n, "deg": deg, "bs": bs}
    if kmax > 1:
        case["k"] = int(round(math.exp(rng.uniform(0, math.log(kmax)))))
    return case


# ------------------------------------------------------------------ graphs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _csr(u, v, n):
    """int32 CSR of the symmetric graph with edges {u, v}."""
    keep = (u != v) & (u < n) & (v < n)
    u, v = u[keep], v[keep]
    key = torch.unique(torch.cat([u * n + v, v * n + u]))
    row = torch.div(key, n, rounding_mode="floor")
    rowptr = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    rowptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0).to(torch.int32)
    return rowptr, (key - row * n).to(torch.int32), row.to(torch.int32)


def _relabel(row, colind, n, gen):
    """The graph with the vertices of each aligned group of 8 renumbered among
    themselves: another graph with as many nonzeros in as many tiles."""
    full = n // 8
    p = torch.arange(n, device=DEV)
    order = torch.rand(full, 8, device=DEV, generator=gen).argsort(1)
    p[:full * 8] = (torch.arange(full, device=DEV)[:, None] * 8 + order).reshape(-1)
    return _csr(p[row.long()], p[colind.long()], n)


def graph(case, seed):
    """(rowptr, colind, row of each entry), int32, on the GPU."""
    n, deg = case["n"], case["deg"]
    gen = _gen(seed)
    if case["op"] in ("pack", "spgemm") and case["graph"] != "king":
        # outputs as long for one seed as for another: the structure is fixed, its numbering drawn
        _, colind, row = graph(dict(case, op="count"), 1)
        return _relabel(row, colind, n, gen)
    if case["graph"] == "king":
        m = math.isqrt(n)
        i = torch.arange(n, device=DEV)
        x, y = i % m, torch.div(i, m, rounding_mode="floor")
        u, v = [], []
        for dx, dy in ((1, 0), (0, 1), (1, 1), (-1, 1)):
            ok = (x + dx >= 0) & (x + dx < m) & (y + dy < m)
            u.append(i[ok])
            v.append(i[ok] + dy * m + dx)
        _, colind, row = _csr(torch.cat(u), torch.cat(v), n)
        # the part of its edges that triangles are counted in, or that components are found in
        part = {"tc": 62, "cc": 24}.get(case["op"])
        if part:
            keep = _weights(row, colind, n, seed) <= part
            colind, row = colind[keep], row[keep]
        return _relabel(row, colind, n, gen)
    if case["graph"] == "er":
        e = torch.randint(0, n, (2, n * deg // 2), device=DEV, generator=gen)
        return _csr(e[0], e[1], n)
    scale = max(1, (n - 1).bit_length())
    m = deg << scale
    a, b, c, _ = RMAT
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        r = torch.rand(m, device=DEV, generator=gen)
        u = 2 * u + (r >= a + b)
        v = 2 * v + (((r >= a) & (r < a + b)) | (r >= a + b + c))
    return _csr(u, v, n)


def _weights(row, col, n, seed):
    """uint32 weight in [1, 64] of each entry, the same in both directions (as int32)."""
    lo, hi = torch.minimum(row, col).to(torch.int64), torch.maximum(row, col).to(torch.int64)
    h = (lo * n + hi + seed) * 0x2545F4914F6CDD1D
    h = (h ^ (h >> 29)) * 0x1B873593CC9E2D51
    return (((h >> 33) & 63) + 1).to(torch.int32)


# ------------------------------------------------------------------ states
def _view(t):
    return gbo.DeviceView(t.data_ptr(), t.numel() * t.element_size())


def _pack(rowptr, colind, n, bs, direction=0):
    return gbo.BsrMatrix.from_device_csr(_view(rowptr), _view(colind), n, n, bs, direction)


def _i32(n):
    return torch.empty(n, dtype=torch.int32, device=DEV)


def _ppr_inputs(n, k, gen):
    """Teleport vectors over a few seed vertices each, and a loss gradient."""
    S = torch.zeros(n, k, device=DEV)
    cnt = min(SEEDS, n)
    at = torch.randperm(n, device=DEV, generator=gen)[:cnt, None] + torch.randint(0, n, (1, k), device=DEV, generator=gen)
    S.scatter_(0, at % n, torch.rand(cnt, k, device=DEV, generator=gen) ** 10 + 1e-6)
    return S / S.sum(0, keepdim=True), torch.randn(n, k, device=DEV, generator=gen)


def prepare(case, seed):
    op, n, bs = case["op"], case["n"], case["bs"]
    rowptr, colind, row = graph(case, seed)
    gen = _gen(seed + 1)
    s = {"op": op, "n": n, "bs": bs}
    if op == "pack":
        s.update(csr=(rowptr, colind), rowptr=_i32((n + bs - 1) // bs + 1))
        return s
    if op in ("tc", "spgemm"):
        # L and L^T; for the general product L is lower by whole groups of 8 (a renumbering moves
        # nothing across them), so that it too is as large for each seed
        r, c = (row // 8, colind // 8) if op == "spgemm" else (row, colind)
        parts = []
        for keep in (r > c, r < c):
            rp = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
            rp[1:] = torch.cumsum(torch.bincount(row[keep], minlength=n), 0).to(torch.int32)
            parts.append((rp, colind[keep].contiguous()))
        s["A"] = _pack(*parts[0], n, bs)
        s["B"] = _pack(*parts[1], n, bs, 1 if op == "tc" else 0)
        return s
    s["A"] = A = _pack(rowptr, colind, n, bs)
    if op == "count":
        x = (torch.rand(n, device=DEV, generator=gen) < 0.5).float()
        s["x"] = torch.zeros((n + bs - 1) // bs, dtype=WORD[bs], device=DEV)
        gbo._check(gbo.lib().gbo_pack_vec(bs, x.data_ptr(), s["x"].data_ptr(), n, None))
        s["y"] = _i32(n)
    elif op == "sum":
        s["x"] = torch.rand(n, device=DEV, generator=gen)
        s["y"] = torch.empty(n, device=DEV)
    elif op == "min":
        s["x"] = torch.randperm(n, device=DEV, generator=gen).to(torch.int32)
        s["y"] = _i32(n)
    if op in ("minplus", "sssp"):
        w = _weights(row, colind, n, seed)
        s["w"], s["woff"] = torch.empty_like(w), torch.empty(A.nblocks + 1, dtype=torch.int64, device=DEV)
        gbo._check(gbo.lib().gbo_csr2bsr_values_u32(A.ref, rowptr.data_ptr(), colind.data_ptr(), w.data_ptr(),
                                                    s["w"].data_ptr(), s["woff"].data_ptr(), None))
    if op == "minplus":  # half of the distances known, as in the middle of a search
        d = torch.randint(0, 1000, (n,), device=DEV, generator=gen, dtype=torch.int32)
        s["x"] = torch.where(torch.rand(n, device=DEV, generator=gen) < 0.5, d, torch.full_like(d, -1))
        s["y"] = _i32(n)
    if op in ("bfs", "bfs_do", "sssp", "cc"):
        s["out"], s["sizes"] = _i32(n), np.zeros(MAX_LEVELS, np.int64)
        # an endpoint of a drawn edge: a search from an isolated vertex is no search
        at = int(torch.randint(0, max(colind.numel(), 1), (1,), device=DEV, generator=gen))
        s["source"] = int(colind[at]) if colind.numel() else 0
    if op == "sssp":
        s["weights"] = _Weights(_view(s["w"]), _view(s["woff"]))
    if op in ("pagerank", "ppr"):
        s["outdeg"] = (rowptr[1:] - rowptr[:-1]).contiguous()
    if op == "pagerank":
        s["out"] = torch.empty(n, device=DEV)
    if op == "msbfs":
        s["sources"] = torch.randint(0, n, (case["k"],), device=DEV, generator=gen).cpu().numpy().astype(np.int32)
        s["out"] = _i32(case["k"] * n)
    if op == "ppr":
        S, s["W"] = _ppr_inputs(n, case["k"], gen)
        s["S"] = S.requires_grad_(True)
        s["alpha"] = torch.tensor(ALPHA, requires_grad=True)
    return s


class _Weights:
    """Per-nonzero weights in tile bit order, held in torch tensors (as gbo.TileValues holds its own)."""

    def __init__(self, tval, woff):
        self.tval, self.woff = tval, woff


# ---------------------------------------------------------------- one pass
def run(s):
    op, A, L = s["op"], s.get("A"), gbo.lib()
    if op == "count":
        gbo._check(L.gbo_bsrbmv_count(A.ref, s["x"].data_ptr(), s["y"].data_ptr(), 0, None))
        return s["y"]
    if op == "sum":
        gbo._check(L.gbo_bsrbmv_sum_f32(A.ref, s["x"].data_ptr(), s["y"].data_ptr(), None))
        return s["y"]
    if op == "min":
        gbo._check(L.gbo_bsrbmv_min_i32(A.ref, s["x"].data_ptr(), s["y"].data_ptr(), None))
        return s["y"]
    if op == "minplus":
        gbo._check(L.gbo_bsrbmv_minplus(A.ref, s["w"].data_ptr(), s["woff"].data_ptr(), s["x"].data_ptr(),
                                        s["y"].data_ptr(), None))
        return s["y"]
    if op in ("bfs", "bfs_do"):
        nl, args = ctypes.c_int32(), (s["source"], s["out"].data_ptr(), s["sizes"].ctypes.data, MAX_LEVELS)
        if op == "bfs":
            gbo._check(L.gbo_bfs(A.ref, *args, ctypes.byref(nl), None))
        else:
            gbo._check(L.gbo_bfs_do(A.ref, A.ref, *args, ctypes.byref(nl), None))
        return s["out"], s["sizes"], nl.value
    if op == "sssp":
        _, iters = gbo.sssp(A, s["source"], s["weights"], out=_view(s["out"]))
        return s["out"], iters
    if op == "pagerank":
        _, iters, _ = gbo.pagerank(A, _view(s["outdeg"]), ALPHA, PR_TOL, 1000, out=_view(s["out"]))
        return s["out"], iters
    if op == "cc":
        _, iters = gbo.cc(A, out=_view(s["out"]))
        return s["out"], iters
    if op == "tc":
        return gbo.bsrbmm_tc(A, s["B"])
    if op == "msbfs":
        levels = gbo.bfs_multisource(A, s["sources"], out=_view(s["out"]))
        return s["out"], levels
    if op == "ppr":
        P = gbo_torch.personalized_pagerank(s["S"], s["alpha"], A, A, s["outdeg"], PPR_TOL, PPR_MAX)
        gS, ga = torch.autograd.grad(P, (s["S"], s["alpha"]), s["W"])
        return P.detach(), gS, ga
    if op == "pack":
        (rowptr, colind), bs, n = s["csr"], s["bs"], s["n"]
        nb = ctypes.c_int64()
        gbo._check(L.gbo_csr2bsr_nnzb_dev(bs, rowptr.data_ptr(), colind.data_ptr(), n, n, s["rowptr"].data_ptr(),
                                          ctypes.byref(nb), None))
        ci, tiles = _i32(nb.value), torch.empty(nb.value * bs, dtype=WORD[bs], device=DEV)
        gbo._check(L.gbo_csr2bsr_fill_dev(bs, 0, rowptr.data_ptr(), colind.data_ptr(), n, n, s["rowptr"].data_ptr(),
                                          ci.data_ptr(), tiles.data_ptr(), None))
        return s["rowptr"], ci, tiles
    if op == "spgemm":
        B, bs = s["B"], s["bs"]
        nb, nnz = ctypes.c_int64(), ctypes.c_int64()
        rp = _i32(A.nblockrows + 1)
        gbo._check(L.gbo_bsrbmm_symbolic(A.ref, B.ref, rp.data_ptr(), ctypes.byref(nb), None))
        ci, tiles = _i32(nb.value), torch.empty(nb.value * bs, dtype=WORD[bs], device=DEV)
        off = torch.empty(nb.value + 1, dtype=torch.int64, device=DEV)
        gbo._check(L.gbo_bsrbmm_numeric(A.ref, B.ref, rp.data_ptr(), nb.value, ci.data_ptr(), tiles.data_ptr(),
                                        off.data_ptr(), ctypes.byref(nnz), None))
        C = gbo.BsrStruct(bs=bs, dir=0, nrows=A.nrows, ncols=B.ncols, nblockrows=A.nblockrows,
                          nblockcols=B.nblockcols, nblocks=nb.value, rowptr=rp.data_ptr(), colind=ci.data_ptr(),
                          tiles=tiles.data_ptr())
        counts = _i32(nnz.value)
        gbo._check(L.gbo_bsrbmm_values(A.ref, B.ref, ctypes.byref(C), off.data_ptr(), counts.data_ptr(), None))
        return rp, ci, tiles, off, counts
    raise ValueError(op)


# --------------------------------------------------------------- 64 bits
def _matrix(rowptr, colind, n):
    return torch.sparse_csr_tensor(rowptr.long(), colind.long(),
                                   torch.ones(colind.numel(), dtype=torch.float64, device=DEV), size=(n, n))


def exact(case, seed):
    """The floating outputs in 64 bits; None in the place of whole numbers."""
    op, n = case["op"], case["n"]
    if op not in ("sum", "pagerank", "ppr"):
        return None
    rowptr, colind, _ = graph(case, seed)
    gen = _gen(seed + 1)
    A = _matrix(rowptr, colind, n)
    if op == "sum":
        x = torch.rand(n, device=DEV, generator=gen).double()
        return (A @ x[:, None])[:, 0]
    deg = (rowptr[1:] - rowptr[:-1]).double()[:, None]
    inv = torch.where(deg > 0, 1.0 / deg.clamp(min=1), torch.zeros_like(deg))
    alpha = float(np.float32(ALPHA))
    if op == "pagerank":
        p = torch.full((n, 1), 1.0 / n, dtype=torch.float64, device=DEV)
        for _ in range(1000):
            q = alpha * (A @ (p * inv)) + (1 - alpha) / n
            delta, p = float((q - p).abs().sum()), q
            if delta < PR_TOL:
                break
        return p[:, 0], None
    S, W = (t.double() for t in _ppr_inputs(n, case["k"], gen))

    def solve(step, x0):
        x, norm = x0, x0.abs().sum(0)
        for _ in range(PPR_MAX):
            y = step(x)
            delta, x = float(((y - x).abs().sum(0) / norm).max()), y
            if delta < PPR_TOL:
                break
        return x

    P = solve(lambda p: alpha * (A @ (p * inv)) + (1 - alpha) * S, S)
    lam = solve(lambda v: alpha * inv * (A @ v) + W, W)
    return P, (1 - alpha) * lam, (lam * (A @ (P * inv) - S)).sum()


# ------------------------------------------------------------------- work
def _tiles(case, bs):
    """Expected nonzeros (bs 1) or tiles of the adjacency matrix."""
    n, deg = case["n"], case["deg"]
    if case["graph"] == "king":
        return 8.0 * n if bs == 1 else 3.0 * n / bs * (1 + 1.0 / min(bs, 32)) + n / bs * 2 * min(1.0, 1.0 * bs / n ** 0.5)
    if case["graph"] == "er":
        cells = (n / bs) ** 2
        return cells * -math.expm1(-n * deg / cells)
    # R-MAT cells at this depth by their numbers of a, b or c, and d steps
    scale = max(1, (n - 1).bit_length())
    d = max(0, scale - int(math.log2(bs)))
    total = 0.0
    for i in range(d + 1):
        for j in range(d + 1 - i):
            cells = math.comb(d, i) * math.comb(d - i, j) * 2.0 ** j
            p = RMAT[0] ** i * RMAT[1] ** j * RMAT[3] ** (d - i - j)
            total += cells * -math.expm1(-2.0 * (deg << scale) * p)
    # the part of the edges that falls inside the cut
    cut = n / (1 << scale)
    return total * min(1.0, cut ** 0.4)


def work(case):
    """Bytes: the packed matrix and the vectors once; operations: one add (or
    min, or) per nonzero, column and iteration.  Tile counts are expected
    values.  What grows with the data (searches, products) counts its inputs
    and outputs alone."""
    op, n, bs, k = case["op"], case["n"], case["bs"], case.get("k", 1)
    nnz, t = _tiles(case, 1), _tiles(case, bs)
    matrix = t * (bs * bs / 8 + 4) + 4 * (n / bs + 1)
    if op == "pack":
        return {"bytes": 4 * nnz + 4 * n + matrix, "flops": nnz}
    if op == "tc":
        return {"bytes": matrix, "flops": nnz}
    if op == "spgemm":
        # C = L L^T, L of whole groups of 8: about 3 values per nonzero of L on the grid, deg on an evenly spread graph
        vals = nnz / 2 * (3 if case["graph"] == "king" else case["deg"])
        ctiles = 1.2 * t if case["graph"] == "king" else vals
        return {"bytes": matrix + ctiles * (bs * bs / 8 + 4 + 8) + 4 * vals, "flops": vals}
    if op == "count":
        return {"bytes": matrix + n / 8 + 4 * n, "flops": nnz}
    if op in ("sum", "min"):
        return {"bytes": matrix + 8 * n, "flops": nnz}
    if op == "minplus":
        return {"bytes": matrix + 8 * n + 4 * nnz + 8 * t, "flops": 2 * nnz}
    if op == "sssp":
        return {"bytes": matrix + 4 * n + 4 * nnz + 8 * t, "flops": 2 * nnz}
    if op == "ppr":
        # S and W in, P and both gradients out, each n x k; about 60 iterations each way at this tolerance
        return {"bytes": matrix + 16 * n * k, "flops": 120 * nnz * k}
    if op == "msbfs":
        return {"bytes": matrix + 4 * n * k, "flops": nnz * k}
    if op == "pagerank":
        return {"bytes": matrix + 8 * n, "flops": 10 * nnz}
    return {"bytes": matrix + 4 * n, "flops": nnz}
