"""The work this library is used for, as timed cases.

Every case is one pass through the public Python entry points on data already
in HBM, with the plan a program would keep.  The kinds:

  pagerank   PageRankPlan.run: one solve from uniform (or one-hot) scores
  spmv       SpmvPlan.run: y <- y + A x
  train      one step of a model with a sparse layer: refresh_values, forward
             y = A x and backward (dA, dx) through torch.autograd
  ppr        PersonalizedPageRankPlan.run: k one-hot seeds at once
  wpr        weighted_pagerank forward and backward through torch.autograd
  multi      MultiGraphPageRank.run: many uneven graphs at once
  symgs      SymGSPlan.run on a 27-point stencil in 8 colors
  build      graph.csr_from_edges_device: an edge list in HBM to a CSR

Inputs are made with plain torch from the seed alone: RMAT graphs (a, b, c, d =
0.57, 0.19, 0.19, 0.05, self-loops and duplicates removed, any number of
vertices), matrices of random sorted distinct columns, stencils.  The sizes of
all results depend on the case alone, not on the seed.
"""
from __future__ import annotations

import math
import random

import torch

import gardenia_ocl_amd as ga
from gardenia_ocl_amd import autograd as ga_autograd
from gardenia_ocl_amd import graph as ga_graph

DEV = "cuda"
DAMP = 0.85


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # config "plain pull PageRank, RMAT scale 16, tol 1e-4": a small graph solved to
        # convergence, ~25 dependent iterations of a few 10 us: latency counts
        {"name": "pr_rmat16", "kind": "pagerank", "m": 65536, "raw": 16 << 16, "tol": 1e-4,
         "iters": 100},
        # a mid-size web or social graph (about a million vertices, no round numbers) to a tight
        # tolerance
        {"name": "pr_mid", "kind": "pagerank", "m": 1000003, "raw": 17000051, "tol": 1e-6,
         "iters": 200},
        # config "RMAT scale 24, 20 fixed iterations": the headline throughput run
        {"name": "pr_rmat24", "kind": "pagerank", "m": 1 << 24, "raw": 16 << 24, "tol": 0.0,
         "iters": 20},
        # the smallest SpMV: one call of an iterative solver on a small system
        {"name": "spmv_small", "kind": "spmv", "rows": 30011, "cols": 30011, "per_row": 21,
         "form": "random", "mode": "tiles"},
        # config "2^22 x 2^22, 32 nonzeros per row in uniform random columns"
        {"name": "spmv_er22", "kind": "spmv", "rows": 1 << 22, "cols": 1 << 22, "per_row": 32,
         "form": "random", "mode": "auto"},
        # a power-law matrix (a weighted graph's adjacency): very uneven rows, the plan's default
        # mode
        {"name": "spmv_powerlaw", "kind": "spmv", "rows": 2500009, "cols": 2500009, "per_row": 16,
         "form": "rmat", "mode": "tiles"},
        # training through a sparse layer: values change every step; rectangular
        {"name": "train_sparse", "kind": "train", "rows": 3000017, "cols": 2000003, "per_row": 16,
         "form": "random", "mode": "auto"},
        # batched personalised PageRank: recommendation scores for a batch of users
        {"name": "ppr_k128", "kind": "ppr", "m": 700001, "raw": 11000003, "k": 128, "tol": 1e-5,
         "iters": 100},
        # config "differentiable weighted PageRank, RMAT scale 20", forward and backward
        {"name": "wpr_rmat20", "kind": "wpr", "m": 1 << 20, "edges": 16000000, "tol": 1e-7,
         "iters": 200},
        # config "64 independent RMAT graphs of uneven scales 12-18 in one launch"
        {"name": "multi_64", "kind": "multi", "graphs": 64, "lo": 1 << 12, "hi": 1 << 18,
         "tol": 1e-4, "iters": 100},
        # the smoother of an HPCG-like multigrid: symmetric Gauss-Seidel on a 27-point stencil
        {"name": "symgs_stencil", "kind": "symgs", "n": 97, "sweeps": 2},
        # graph construction on the device: raw RMAT edges (repeats and self-loops among them) to
        # a PageRank in-CSR
        {"name": "build_rmat22", "kind": "build", "m": 1 << 22, "edges": 60000000,
         "weights": False, "symmetrize": False, "transpose": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pagerank", "pagerank", "pagerank", "spmv", "spmv", "spmv", "train", "ppr",
                       "wpr", "multi", "symgs", "build"])
    if kind == "pagerank":
        m = _log_int(rng, 2000, 1 << 23)
        tol = rng.choice([0.0, 1e-3, 1e-4, 1e-6])
        raw = min(m * rng.randint(4, 32), 1 << (26 if tol else 27))
        return {"kind": kind, "m": m, "raw": raw, "tol": tol, "iters": 20 if tol == 0.0 else 200}
    if kind in ("spmv", "train"):
        top = 1 << 22 if kind == "spmv" else 3 << 20
        rows = _log_int(rng, 5000, top)
        per_row = rng.randint(3, 40)
        form = "random" if kind == "train" else rng.choice(["random", "rmat"])
        cols = rows if form == "rmat" else _log_int(rng, max(5000, rows // 4),
                                                     min(top, rows * 4))
        per_row = max(1, min(per_row, (1 << 26) // rows))
        return {"kind": kind, "rows": rows, "cols": cols, "per_row": per_row, "form": form,
                "mode": rng.choice(["tiles", "auto"])}
    if kind == "ppr":
        m = _log_int(rng, 3000, 300000)
        return {"kind": kind, "m": m, "raw": m * rng.randint(6, 20), "k": 64 * rng.randint(1, 4),
                "tol": rng.choice([1e-3, 1e-4, 1e-5]), "iters": 100}
    if kind == "wpr":
        m = _log_int(rng, 5000, 1 << 20)
        return {"kind": kind, "m": m, "edges": m * rng.randint(4, 14),
                "tol": rng.choice([1e-5, 1e-6, 1e-7]), "iters": 200}
    if kind == "multi":
        lo = _log_int(rng, 500, 5000)
        return {"kind": kind, "graphs": rng.randint(5, 60), "lo": lo,
                "hi": lo * rng.randint(4, 40), "tol": rng.choice([1e-3, 1e-4, 1e-5]),
                "iters": 100}
    if kind == "symgs":
        return {"kind": kind, "n": rng.randint(16, 128), "sweeps": rng.randint(1, 3)}
    m = _log_int(rng, 5000, 1 << 22)
    return {"kind": "build", "m": m, "edges": m * rng.randint(4, 12),
            "weights": rng.random() < 0.5, "symmetrize": rng.random() < 0.3,
            "transpose": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs (plain torch)

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2654435761 % (1 << 31) + 12345)
    return g


def _rmat_edges(m, raw, gen):
    """Raw RMAT edges (src, dst) int64 over m vertices."""
    scale = max(1, (m - 1).bit_length())
    a, ab, abc = 0.57, 0.76, 0.95
    src = torch.empty(raw, dtype=torch.int64, device=DEV)
    dst = torch.empty(raw, dtype=torch.int64, device=DEV)
    step = 1 << 25
    for o in range(0, raw, step):
        n = min(step, raw - o)
        s = torch.zeros(n, dtype=torch.int32, device=DEV)
        d = torch.zeros(n, dtype=torch.int32, device=DEV)
        for _ in range(scale):
            r = torch.rand(n, generator=gen, device=DEV)
            s = s * 2 + (r >= ab).int()
            d = d * 2 + (((r >= a) & (r < ab)) | (r >= abc)).int()
        src[o:o + n] = (s.long() * m) >> scale  # any vertex count, same skew
        dst[o:o + n] = (d.long() * m) >> scale
    return src, dst


def _csr(rows, cols, r, c, nnz=None):
    """Sorted CSR (int32 offsets and columns) without duplicates; nnz: that many of the entries,
    evenly spread."""
    key = torch.sort(r * cols + c).values
    keep = torch.ones(key.shape[0], dtype=torch.bool, device=DEV)
    keep[1:] = key[1:] != key[:-1]
    key = key[keep]
    del keep
    if nnz is not None:
        assert key.shape[0] >= nnz, "too many repeated edges"
        key = key[torch.arange(nnz, device=DEV) * key.shape[0] // nnz]
    first = torch.arange(rows + 1, dtype=torch.int64, device=DEV) * cols
    off = torch.searchsorted(key, first).int()
    return off, (key % cols).int()


def _rmat_graph(m, raw, gen, nnz=None):
    """In-CSR (rows = destinations) and out-degrees of an RMAT graph."""
    s, d = _rmat_edges(m, raw, gen)
    keep = s != d
    off, col = _csr(m, m, d[keep], s[keep], nnz)
    deg = torch.bincount(col, minlength=m).int()
    return off, col, deg


def _pm1(n, gen):
    return torch.rand(n, generator=gen, device=DEV) * 2 - 1


def _matrix(case, gen):
    rows, cols, k = case["rows"], case["cols"], case["per_row"]
    if case["form"] == "rmat":
        c, r = _rmat_edges(rows, rows * k, gen)
        off, col = _csr(rows, cols, r, c)
    else:  # entry j of a row: uniform in the j-th of k equal ranges of columns
        j = torch.arange(k, device=DEV)
        lo, hi = j * cols // k, (j + 1) * cols // k
        u = torch.rand((rows, k), generator=gen, device=DEV)
        col = (lo + torch.minimum((u * (hi - lo)).long(), hi - lo - 1)).int().flatten()
        off = torch.arange(rows + 1, device=DEV).mul_(k).int()
    return off, col, _pm1(col.shape[0], gen)


def _stencil(n):
    """27-point stencil on n^3 points: CSR, values, rows in 8-color order, color offsets."""
    m = n ** 3
    i = torch.arange(m, device=DEV)
    x, y, z = i % n, (i // n) % n, i // (n * n)
    keep, cols = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                keep.append((x + dx >= 0) & (x + dx < n) & (y + dy >= 0) & (y + dy < n)
                            & (z + dz >= 0) & (z + dz < n))
                cols.append(i + dz * n * n + dy * n + dx)
    keep, cols = torch.stack(keep, 1), torch.stack(cols, 1)
    col = cols[keep]
    rows = i[:, None].expand(-1, 27)[keep]
    off = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(keep.sum(1), 0)
    lo, hi = torch.minimum(rows, col), torch.maximum(rows, col)
    val = torch.where(rows == col, 26.5, -(0.5 + ((lo * 7919 + hi * 104729) % 1000) / 2000.0))
    color = (x % 2) + 2 * (y % 2) + 4 * (z % 2)
    order = torch.sort(color, stable=True).indices
    co = [0] + torch.cumsum(torch.bincount(color, minlength=8), 0).tolist()
    return off.int(), col.int(), val.float(), order.int(), co


def _edge_list(case, gen):
    """A raw edge list in random order: `edges` different edges (of a symmetric graph: each
    undirected edge once), a tenth of them twice, and a few self-loops."""
    m, n = case["m"], case["edges"]
    s, d = _rmat_edges(m, 2 * n, gen)
    if case["symmetrize"]:
        s, d = torch.minimum(s, d), torch.maximum(s, d)
    keep = s != d
    off, col = _csr(m, m, s[keep], d[keep], n)
    s = torch.repeat_interleave(torch.arange(m, device=DEV), torch.diff(off.long()))
    again = torch.randint(0, n, (n // 10,), generator=gen, device=DEV)
    loops = torch.randint(0, m, (n // 100,), generator=gen, device=DEV)
    s, d = torch.cat([s, s[again], loops]), torch.cat([col.long(), col[again].long(), loops])
    order = torch.randperm(s.shape[0], generator=gen, device=DEV)
    return s[order].int(), d[order].int()


def _multi_sizes(case):
    r = random.Random(case["lo"] * 7 + case["graphs"])
    return [_log_int(r, case["lo"], case["hi"]) for _ in range(case["graphs"])]


def _inputs(case, seed):
    """Everything random of a case, by name."""
    gen, kind = _gen(seed), case["kind"]
    if kind == "pagerank":
        off, col, deg = _rmat_graph(case["m"], case["raw"], gen)
        return {"off": off, "col": col, "deg": deg}
    if kind in ("spmv", "train"):
        off, col, val = _matrix(case, gen)
        return {"off": off, "col": col, "val": val, "x": _pm1(case["cols"], gen),
                "g": _pm1(case["rows"], gen)}
    if kind == "ppr":
        off, col, deg = _rmat_graph(case["m"], case["raw"], gen)
        live = torch.nonzero(deg > 0).flatten()
        pick = torch.randint(0, live.shape[0], (case["k"],), generator=gen, device=DEV)
        return {"off": off, "col": col, "deg": deg, "seeds": live[pick].int()}
    if kind == "wpr":
        off, col, _ = _rmat_graph(case["m"], 2 * case["edges"], gen, case["edges"])
        w = torch.rand(col.shape[0], generator=gen, device=DEV) + 0.5
        return {"off": off, "col": col, "w": w,
                "g": torch.randn(case["m"], generator=gen, device=DEV)}
    if kind == "multi":
        return {"graphs": [_rmat_graph(m, 16 * m, gen) for m in _multi_sizes(case)]}
    if kind == "symgs":
        off, col, val, order, co = _stencil(case["n"])
        return {"off": off, "col": col, "val": val, "order": order, "co": co,
                "b": _pm1(case["n"] ** 3, gen)}
    s, d = _edge_list(case, gen)
    w = torch.rand(s.shape[0], generator=gen, device=DEV) if case["weights"] else None
    return {"src": s, "dst": d, "w": w}


# ------------------------------------------------------------------ the calls

def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"], kind = case, case["kind"]
    if kind == "pagerank":
        st["plan"] = ga.PageRankPlan(st["off"], st["col"], st["deg"])
        st["scores"] = torch.empty(case["m"], dtype=torch.float32, device=DEV)
    elif kind == "spmv":
        st["plan"] = ga.SpmvPlan(st["off"], st["col"], st["val"], case["cols"], mode=case["mode"])
        st["y"] = torch.empty(case["rows"], dtype=torch.float32, device=DEV)
    elif kind == "train":
        st["val"].requires_grad_(True)
        st["x"].requires_grad_(True)
        st["plan"] = ga.SpmvPlan(st["off"], st["col"], st["val"].detach(), case["cols"],
                                 mode=case["mode"])
        st["bwd"] = ga_autograd.SpmvBackwardPlan(st["off"], st["col"], case["cols"])
    elif kind == "ppr":
        st["plan"] = ga.PersonalizedPageRankPlan(st["off"], st["col"], st["deg"], case["k"])
    elif kind == "wpr":
        st["w"].requires_grad_(True)
        st["plan"] = ga_autograd.WeightedPageRankPlan(st["off"], st["col"], st["w"].detach())
    elif kind == "multi":
        sizes = [g[2].shape[0] for g in st["graphs"]]
        st["plan"] = ga.MultiGraphPageRank(st["graphs"])
        st["init"] = torch.cat([torch.full((m,), 1.0 / m, device=DEV) for m in sizes])
        st["flat"] = torch.empty_like(st["init"])
        st["scores"] = list(torch.split(st["flat"], sizes))
        del st["graphs"]  # the plan keeps its own copy
    elif kind == "symgs":
        st["plan"] = ga.SymGSPlan(st["off"], st["col"], st["val"], st["order"], st["co"])
        st["x"] = torch.empty(case["n"] ** 3, dtype=torch.float32, device=DEV)
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "pagerank":
        st["scores"].fill_(1.0 / case["m"])
        stats, errs = st["plan"].run(st["scores"], tol=case["tol"], max_iter=case["iters"])
        return {"scores": st["scores"], "iterations": stats["iterations"], "l1": float(errs[-1])}
    if kind == "spmv":
        st["y"].zero_()
        st["plan"].run(st["x"], st["y"])
        return st["y"]
    if kind == "train":
        st["plan"].refresh_values()  # the optimizer changed the values
        y = ga_autograd.spmv(st["val"], st["x"], st["plan"], st["bwd"])
        dA, dx = torch.autograd.grad(y, (st["val"], st["x"]), st["g"])
        return {"y": y.detach(), "dA": dA, "dx": dx}
    if kind == "ppr":
        X = st["plan"].one_hot(st["seeds"])
        stats, _, col_l1 = st["plan"].run(st["seeds"], X, tol=case["tol"], max_iter=case["iters"])
        return {"X": X, "iterations": st["plan"].column_iterations(), "l1": col_l1}
    if kind == "wpr":
        x = ga_autograd.weighted_pagerank(st["w"], st["plan"], tol=case["tol"],
                                          max_iter=case["iters"])
        (grad,) = torch.autograd.grad(x, st["w"], st["g"])
        return {"x": x.detach(), "grad": grad}
    if kind == "multi":
        st["flat"].copy_(st["init"])
        its, errs, _ = st["plan"].run(st["scores"], tol=case["tol"], max_iter=case["iters"])
        return {"scores": st["flat"], "iterations": its, "l1": errs}
    if kind == "symgs":
        st["x"].zero_()
        st["plan"].run(st["x"], st["b"], case["sweeps"])
        return st["x"]
    return ga_graph.csr_from_edges_device(
        case["m"], st["src"], st["dst"], st["w"], symmetrize=case["symmetrize"],
        transpose=case["transpose"])


# ------------------------------------------------------------------ necessary work

def _iterations(case):
    """Iterations a solve takes: fixed, or the usual decay of the L1 change per iteration on these
    graphs (a factor of about 0.74)."""
    if case["tol"] == 0.0:
        return case["iters"]
    return min(case["iters"], math.ceil(math.log(case["tol"]) / math.log(0.74)))


def work(case):
    kind = case["kind"]
    if kind == "pagerank":
        m, e = case["m"], case["raw"]
        it = _iterations(case)
        return {"bytes": it * (4 * e + 24 * m), "flops": it * (e + 4 * m)}
    if kind in ("spmv", "train"):
        r, c = case["rows"], case["cols"]
        nnz = r * case["per_row"]
        if kind == "spmv":
            return {"bytes": 8 * nnz + 12 * r + 4 * c, "flops": 2 * nnz}
        # indices and values once, dA once; offsets, x, g, y, dx
        return {"bytes": 12 * nnz + 12 * r + 8 * c, "flops": 5 * nnz}
    if kind == "ppr":
        it = _iterations(case) / 2  # columns stop one by one
        m, e, k = case["m"], case["raw"], case["k"]
        return {"bytes": it * (4 * e + 8 * m + 16 * m * k), "flops": it * k * (e + 4 * m)}
    if kind == "wpr":
        m, e = case["m"], case["edges"]
        it = 3 * _iterations(case)  # the adjoint takes about twice the forward's iterations
        return {"bytes": it * (8 * e + 24 * m) + 16 * e, "flops": it * 2 * e}
    if kind == "multi":
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        m = int(case["graphs"] * mean)
        it = _iterations(case)
        return {"bytes": it * (4 * 16 * m + 24 * m), "flops": it * 20 * m}
    if kind == "symgs":
        m = case["n"] ** 3
        return {"bytes": 2 * case["sweeps"] * (8 * 26 * m + 20 * m),
                "flops": 2 * case["sweeps"] * 54 * m}
    e = case["edges"] * (2 if case["symmetrize"] else 1)
    n = case["edges"] * 1.11
    return {"bytes": n * (12 if case["weights"] else 8) + e * 8 + 8 * case["m"], "flops": 0}


# ------------------------------------------------------------------ 64-bit results

def _sparse(off, col, val, rows, cols):
    return torch.sparse_csr_tensor(off.long(), col.long(), val.double(), (rows, cols))


def _exact_pr(off, col, deg, tol, iters):
    m = deg.shape[0]
    inv = 1.0 / deg.double().clamp(min=1.0)
    A = _sparse(off, col, inv[col.long()], m, m)
    x = torch.full((m,), 1.0 / m, dtype=torch.float64, device=DEV)
    log = []
    for _ in range(iters):
        nx = (1.0 - DAMP) / m + DAMP * (A @ x)
        log.append(float((nx - x).abs().sum()))
        x = nx
        if log[-1] < tol:
            break
    return x, log


def exact(case, seed):
    kind = case["kind"]
    if kind == "build":
        return None  # whole numbers, and weights that are copied
    st = _inputs(case, seed)
    if kind == "pagerank":
        x, _ = _exact_pr(st["off"], st["col"], st["deg"], case["tol"], case["iters"])
        return {"scores": x, "iterations": None, "l1": None}
    if kind in ("spmv", "train"):
        off, col, val, x = st["off"], st["col"], st["val"].double(), st["x"].double()
        rows, cols = case["rows"], case["cols"]
        y = _sparse(off, col, val, rows, cols) @ x
        if kind == "spmv":
            return y
        row = torch.repeat_interleave(torch.arange(rows, device=DEV), torch.diff(off.long()))
        gr = st["g"].double()[row]
        dx = torch.zeros(cols, dtype=torch.float64, device=DEV)
        dx.index_add_(0, col.long(), val * gr)
        return {"y": y, "dA": gr * x[col.long()], "dx": dx}
    if kind == "ppr":
        m, k = case["m"], case["k"]
        inv = 1.0 / st["deg"].double().clamp(min=1.0)
        A = _sparse(st["off"], st["col"], inv[st["col"].long()], m, m)
        seeds, lanes = st["seeds"].long(), torch.arange(k, device=DEV)
        X = torch.zeros((m, k), dtype=torch.float64, device=DEV)
        X[seeds, lanes] = 1.0
        live = torch.ones(k, dtype=torch.bool, device=DEV)
        for _ in range(case["iters"]):
            N = DAMP * (A @ X)
            N[seeds, lanes] += 1.0 - DAMP
            change = (N - X).abs().sum(0)
            X = torch.where(live[None, :], N, X)
            live &= change >= case["tol"]
            if not bool(live.any()):
                break
        return {"X": X, "iterations": None, "l1": None}
    if kind == "wpr":
        m, off, col, w = case["m"], st["off"], st["col"].long(), st["w"].double()
        row = torch.repeat_interleave(torch.arange(m, device=DEV), torch.diff(off.long()))
        s = torch.zeros(m, dtype=torch.float64, device=DEV).index_add_(0, col, w)
        p = w / s[col]
        A = _sparse(off, col, p, m, m)
        x = torch.full((m,), 1.0 / m, dtype=torch.float64, device=DEV)
        for _ in range(case["iters"]):
            nx = (1.0 - DAMP) / m + DAMP * (A @ x)
            change = float((nx - x).abs().sum())
            x = nx
            if change < case["tol"]:
                break
        order = torch.sort(col, stable=True).indices
        toff = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
        toff[1:] = torch.cumsum(torch.bincount(col, minlength=m), 0)
        At = _sparse(toff, row[order], p[order], m, m)
        g = st["g"].double()
        lam = g.clone()
        for _ in range(case["iters"]):
            nl = g + DAMP * (At @ lam)
            change = float((nl - lam).abs().sum())
            lam = nl
            if change < case["tol"]:
                break
        q = At @ lam
        xs = torch.where(s > 0, x / s, torch.zeros_like(x))
        return {"x": x, "grad": DAMP * xs[col] * (lam[row] - q[col])}
    if kind == "multi":
        xs = [_exact_pr(off, col, deg, case["tol"], case["iters"])[0]
              for off, col, deg in st["graphs"]]
        return {"scores": torch.cat(xs), "iterations": None, "l1": None}
    # symgs: color by color; rows of one color do not meet
    m = case["n"] ** 3
    off, col, val = st["off"].long(), st["col"].long(), st["val"].double()
    row = torch.repeat_interleave(torch.arange(m, device=DEV), torch.diff(off))
    parts = []
    rank = torch.empty(m, dtype=torch.int64, device=DEV)
    for c in range(8):
        rows = st["order"][st["co"][c]:st["co"][c + 1]].long()
        rank.fill_(-1)
        rank[rows] = torch.arange(rows.shape[0], device=DEV)
        mine = (rank[row] >= 0) & (row != col)
        diag = torch.empty(rows.shape[0], dtype=torch.float64, device=DEV)
        on = (rank[row] >= 0) & (row == col)
        diag[rank[row[on]]] = val[on]
        parts.append((rows, rank[row[mine]], col[mine], val[mine], diag))
    x, b = torch.zeros(m, dtype=torch.float64, device=DEV), st["b"].double()
    for _ in range(case["sweeps"]):
        for c in list(range(8)) + list(range(7, -1, -1)):
            rows, at, cj, v, d = parts[c]
            acc = torch.zeros(rows.shape[0], dtype=torch.float64, device=DEV)
            acc.index_add_(0, at, v * x[cj])
            x[rows] = (b[rows] - acc) / d
    return x
