"""Workloads of the graph engine for timing, through its public entry points.

A case names an operation, a graph family with its sizes, and the options of
the call.  The graphs are the two families of the benchmark and the serving
pool: R-MAT (a/b/c/d = .57/.19/.19/.05, edge factor 16 by default) and 2D
lattices (10 % of the edges removed, 0.1 % long-range edges added), both
undirected, made on the GPU from the seed and built by apspie_graph_from_coo
from device memory.  A vertex count that is not a power of two scales the
R-MAT ids down onto it.  Traversal weights are integers 1..255, products and
SpMSpV values are floats in (0, 1].

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  a graph resident in HBM, sources, result arrays
    run(state)           one call; results stay in HBM
    work(case)           bytes a call cannot do without (inputs + outputs)
    exact(case, seed)    float results in 64 bits, by plain torch
"""
from __future__ import annotations

import ctypes as C
import math

import torch

import apspie_amd as A

DEV = "cuda:0"
RMAT_A, RMAT_B, RMAT_C = 0.57, 0.19, 0.19


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one query on a small graph: latency (the CPU-runnable configuration)
        {"name": "bfs_rmat14", "op": "bfs", "graph": "rmat", "m": 1 << 14, "ef": 16},
        # the headline traversal
        {"name": "bfs_rmat22", "op": "bfs", "graph": "rmat", "m": 1 << 22, "ef": 16},
        # a road-like graph: many narrow levels
        {"name": "bfs_lattice2048", "op": "bfs", "graph": "lattice", "width": 2048},
        # weighted paths on the headline graph
        {"name": "sssp_rmat22", "op": "sssp", "graph": "rmat", "m": 1 << 22, "ef": 16},
        # weighted paths on a mid-size road-like graph of the serving pool
        {"name": "sssp_lattice1024", "op": "sssp", "graph": "lattice", "width": 1024},
        # independent set on the benchmark's graph
        {"name": "mis_rmat20", "op": "mis", "graph": "rmat", "m": 1 << 20, "ef": 16},
        # triangle count with per-vertex counts, the serving pool's size
        {"name": "tc_rmat18", "op": "tc", "graph": "rmat", "m": 1 << 18, "ef": 16},
        # general sparse product A * A, the benchmark's size
        {"name": "spgemm_rmat14", "op": "spgemm", "graph": "rmat", "m": 1 << 14, "ef": 16},
        # one masked (+, x) step from a sparse frontier: a caller's own algorithm
        {"name": "spmspv_rmat18", "op": "spmspv", "graph": "rmat", "m": 1 << 18, "ef": 16,
         "nx": 2621, "semiring": A.SR_PLUS_TIMES, "mask": True},
        # a full batch of the query server on a road-like graph
        {"name": "bfs_batch_lattice2048", "op": "bfs_batch", "graph": "lattice", "width": 2048,
         "nsrc": 128},
        # a small batch of weighted queries
        {"name": "sssp_batch_lattice2048", "op": "sssp_batch", "graph": "lattice",
         "width": 2048, "nsrc": 32},
        # admission: a weighted undirected graph built from device triples
        {"name": "build_rmat20", "op": "build", "graph": "rmat", "m": 1 << 20, "ef": 16,
         "symmetrize": True, "weighted": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["bfs", "bfs", "sssp", "sssp", "mis", "tc", "spgemm", "spmspv",
                     "bfs_batch", "sssp_batch", "build"])
    if op == "bfs" or op == "sssp":
        if rng.random() < 0.5:
            m = _log_int(rng, 1 << 12, 1 << 22)
            return {"op": op, "graph": "rmat", "m": m, "ef": rng.randint(8, 16)}
        return {"op": op, "graph": "lattice",
                "width": _log_int(rng, 64, 2048 if op == "bfs" else 1024)}
    if op == "mis":
        if rng.random() < 0.7:
            return {"op": op, "graph": "rmat", "m": _log_int(rng, 1 << 12, 1 << 20),
                    "ef": rng.randint(8, 16)}
        return {"op": op, "graph": "lattice", "width": _log_int(rng, 64, 1024)}
    if op == "tc":
        return {"op": op, "graph": "rmat", "m": _log_int(rng, 1 << 12, 1 << 18),
                "ef": rng.randint(8, 16)}
    if op == "spgemm":
        if rng.random() < 0.7:
            return {"op": op, "graph": "rmat", "m": _log_int(rng, 1 << 10, 1 << 14),
                    "ef": rng.randint(4, 16)}
        return {"op": op, "graph": "lattice", "width": _log_int(rng, 64, 1024)}
    if op == "spmspv":
        m = _log_int(rng, 1 << 12, 1 << 20)
        return {"op": op, "graph": "rmat", "m": m, "ef": rng.randint(8, 16),
                "nx": max(1, _log_int(rng, 4, m // 8)), "semiring": rng.randint(0, 3),
                "mask": rng.random() < 0.5}
    if op == "bfs_batch":
        if rng.random() < 0.6:
            return {"op": op, "graph": "lattice", "width": _log_int(rng, 128, 2048),
                    "nsrc": _log_int(rng, 4, 128)}
        return {"op": op, "graph": "rmat", "m": _log_int(rng, 1 << 12, 1 << 20),
                "ef": rng.randint(8, 16), "nsrc": _log_int(rng, 4, 128)}
    if op == "sssp_batch":
        if rng.random() < 0.6:
            return {"op": op, "graph": "lattice", "width": _log_int(rng, 128, 2048),
                    "nsrc": _log_int(rng, 4, 32)}
        return {"op": op, "graph": "rmat", "m": _log_int(rng, 1 << 12, 1 << 18),
                "ef": rng.randint(8, 16), "nsrc": _log_int(rng, 4, 32)}
    return {"op": "build", "graph": "rmat", "m": _log_int(rng, 1 << 12, 1 << 20),
            "ef": rng.randint(8, 16), "symmetrize": rng.random() < 0.7,
            "weighted": rng.random() < 0.6}


# ------------------------------------------------------------------ inputs
def _rmat(gen, m, ef):
    scale = max(1, (m - 1).bit_length())
    ne = ef * m
    u = torch.zeros(ne, dtype=torch.int32, device=DEV)
    v = torch.zeros(ne, dtype=torch.int32, device=DEV)
    ab, abc = RMAT_A + RMAT_B, RMAT_A + RMAT_B + RMAT_C
    for _ in range(scale):
        r = torch.rand(ne, generator=gen, device=DEV)
        u = u * 2 + (r >= ab)
        v = v * 2 + (((r >= RMAT_A) & (r < ab)) | (r >= abc))
    if m != 1 << scale:
        u = ((u.long() * m) >> scale).int()
        v = ((v.long() * m) >> scale).int()
    return u, v


def _lattice(gen, w):
    ids = torch.arange(w * w, dtype=torch.int32, device=DEV).view(w, w)
    u = torch.cat([ids[:, :-1].reshape(-1), ids[:-1].reshape(-1)])
    v = torch.cat([ids[:, 1:].reshape(-1), ids[1:].reshape(-1)])
    ne = u.numel()
    keep = torch.rand(ne, generator=gen, device=DEV) >= 0.1
    far = torch.randint(0, w * w, (2, max(1, ne // 1000)), generator=gen, device=DEV,
                        dtype=torch.int32)
    return torch.cat([u[keep], far[0]]), torch.cat([v[keep], far[1]])


def _weights(u, v, seed, whole):
    """One value per undirected edge, whichever way round it is listed."""
    p, q = torch.minimum(u, v).long(), torch.maximum(u, v).long()
    h = (p * 0x9E3779B1 + q * 0x85EBCA6B + (seed % 65521) * 0xC2B2AE35) & 0xFFFFFFFF
    h = ((h ^ (h >> 15)) * 0x2C1B3C6D) & 0xFFFFFFFF
    h = h ^ (h >> 12)
    if whole:
        return (h % 255 + 1).float()
    return ((h & 0xFFFFFF) + 1).float() / float(1 << 24)


def _vertices(case):
    return case["m"] if case["graph"] == "rmat" else case["width"] ** 2


def _edges(case, seed):
    """(u, v, w) of the undirected edges, and the generator for what follows."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1_000_003 * (seed % 1_000_003) + 17)
    u, v = (_rmat(gen, case["m"], case["ef"]) if case["graph"] == "rmat"
            else _lattice(gen, case["width"]))
    w = None
    if case["op"] in ("sssp", "sssp_batch"):
        w = _weights(u, v, seed, True)
    elif case["op"] in ("spgemm", "spmspv") or case.get("weighted"):
        w = _weights(u, v, seed, False)
    return u, v, w, gen


def _connected(u, v, m, k, gen):
    """k distinct vertices with a neighbour, uniform."""
    deg = torch.zeros(m, dtype=torch.int32, device=DEV)
    one = torch.ones_like(u)
    off = (u != v).int() * one
    deg.index_add_(0, u, off)
    deg.index_add_(0, v, off)
    verts = torch.nonzero(deg).view(-1)
    k = min(k, verts.numel())
    return verts[torch.randperm(verts.numel(), generator=gen, device=DEV)[:k]].cpu()


def _frontier(case, gen):
    """Sorted distinct frontier vertices, their values, and the visited mask."""
    m = case["m"]
    xi = torch.randperm(m, generator=gen, device=DEV)[:case["nx"]].int().sort().values
    xv = 1.0 - torch.rand(xi.numel(), generator=gen, device=DEV)
    mask = (torch.rand(m, generator=gen, device=DEV) < 0.5).int() if case["mask"] else None
    return xi, xv, mask


_context = None


def _ctx():
    global _context
    if _context is None:
        _context = A.Context(0)
    return _context


def _build(u, v, w, m, symmetrize=1):
    ctx = _ctx()
    coo = A._Coo(m, m, u.numel(), u.data_ptr(), v.data_ptr(), None if w is None else w.data_ptr())
    h = C.c_void_p()
    A._check(A.lib().apspie_graph_from_coo(ctx.h, C.byref(coo), A.DEVICE, symmetrize,
                                           C.byref(h)), ctx.h)
    return A.Graph(ctx, h)


def _room(case):
    """Entries that a result graph of the case can have, at most."""
    m = _vertices(case)
    if case["op"] == "build":
        return case["ef"] * m * (2 if case["symmetrize"] else 1)
    if case["graph"] == "lattice":  # rows of about four entries, squared
        return 20 * m
    return m * m if m <= 4096 else m * m // 2  # 15 % full at 2^14 vertices


def _csr_room(case):
    """The caller's arrays for a result graph (zero past its entries)."""
    n = _room(case)
    return {"rowptr": torch.zeros(_vertices(case) + 1, dtype=torch.int32, device=DEV),
            "col": torch.zeros(n, dtype=torch.int32, device=DEV),
            "val": torch.zeros(n, dtype=torch.float32, device=DEV)}


def prepare(case, seed):
    ctx = _ctx()
    op, m = case["op"], _vertices(case)
    u, v, w, gen = _edges(case, seed)
    if op == "build":
        st = {"case": case, "ctx": ctx, "u": u, "v": v, "w": w, "m": m, **_csr_room(case)}
        torch.cuda.synchronize()
        return st
    st = {"case": case, "ctx": ctx, "m": m}
    if op in ("bfs", "sssp"):
        st["source"] = int(_connected(u, v, m, 1, gen)[0])
        st["out"] = torch.empty(m, dtype=torch.int32 if op == "bfs" else torch.float32,
                                device=DEV)
    elif op in ("bfs_batch", "sssp_batch"):
        st["sources"] = _connected(u, v, m, case["nsrc"], gen).int().numpy()
        st["out"] = torch.empty(len(st["sources"]), m, device=DEV,
                                dtype=torch.int32 if op == "bfs_batch" else torch.float32)
    elif op in ("mis", "tc"):
        st["out"] = torch.empty(m, dtype=torch.int32, device=DEV)
    elif op == "spmspv":
        st["xi"], st["xv"], st["mask"] = _frontier(case, gen)
        st["yi"] = torch.zeros(m, dtype=torch.int32, device=DEV)
        st["yv"] = torch.zeros(m, dtype=torch.float32, device=DEV)
    elif op == "spgemm":
        st.update(_csr_room(case))
    torch.cuda.synchronize()  # the library runs on its own stream
    st["graph"] = _build(u, v, w, m)
    return st


# --------------------------------------------------------------------- run
def _copy_out(st, g):
    """The CSR arrays of a new graph, copied into the caller's own."""
    view = A._Csr()
    A._check(A.lib().apspie_graph_view(g.h, C.byref(view)))
    L, h = A.lib(), st["ctx"].h
    A._check(L.apspie_memcpy(h, st["rowptr"].data_ptr(), view.rowptr, 4 * (view.m + 1), 2), h)
    if view.nnz > st["col"].numel():
        raise RuntimeError(f"{view.nnz} entries, room for {st['col'].numel()}")
    if view.nnz:
        A._check(L.apspie_memcpy(h, st["col"].data_ptr(), view.col, 4 * view.nnz, 2), h)
        A._check(L.apspie_memcpy(h, st["val"].data_ptr(), view.val, 4 * view.nnz, 2), h)
    return {"rowptr": st["rowptr"], "col": st["col"], "val": st["val"], "nnz": view.nnz}


def run(st):
    case, ctx = st["case"], st["ctx"]
    op = case["op"]
    if op == "bfs":
        ctx.bfs(st["graph"], st["source"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return st["out"]
    if op == "sssp":
        ctx.sssp(st["graph"], st["source"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return st["out"]
    if op == "bfs_batch":
        ctx.bfs_batch(st["graph"], st["sources"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return st["out"]
    if op == "sssp_batch":
        ctx.sssp_batch(st["graph"], st["sources"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return st["out"]
    if op == "mis":
        ctx.mis(st["graph"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return st["out"]
    if op == "tc":
        total, _ = ctx.tc(st["graph"], out=st["out"].data_ptr(), mem=A.DEVICE)
        return {"total": total, "per_row": st["out"]}
    if op == "spgemm":
        g = ctx.spgemm(st["graph"], st["graph"])
        out = _copy_out(st, g)
        g.close()
        return out
    if op == "spmspv":
        ny = C.c_int64()
        mask = st["mask"]
        A._check(A.lib().apspie_spmspv(ctx.h, st["graph"].h, case["semiring"], st["xi"].numel(),
                                       st["xi"].data_ptr(), st["xv"].data_ptr(),
                                       None if mask is None else mask.data_ptr(), C.byref(ny),
                                       st["yi"].data_ptr(), st["yv"].data_ptr(), A.DEVICE,
                                       A.PATH_AUTO), ctx.h)
        return {"ind": st["yi"], "val": st["yv"], "count": ny.value}
    g = _build(st["u"], st["v"], st["w"], st["m"], int(case["symmetrize"]))
    out = _copy_out(st, g)
    g.close()
    return out


# -------------------------------------------------------------------- work
def _entries(case):
    """Stored entries of the symmetric CSR, about (R-MAT repeats ~5 % of its
    edges at scale 22 and more on small graphs)."""
    if case["graph"] == "lattice":
        return int(3.6 * case["width"] ** 2)
    return int(2 * case["ef"] * case["m"] * (0.7 + 0.25 * min(1.0, math.log2(case["m"]) / 22)))


def work(case):
    op, m, nnz = case["op"], _vertices(case), _entries(case)
    csr = 4 * (m + 1) + 4 * nnz
    if op in ("bfs", "mis", "tc"):
        return {"bytes": csr + 4 * m, "flops": 0}
    if op == "sssp":
        return {"bytes": csr + 4 * nnz + 4 * m, "flops": 0}
    if op == "bfs_batch":
        return {"bytes": csr + 4 * m * case["nsrc"], "flops": 0}
    if op == "sssp_batch":
        return {"bytes": csr + 4 * nnz + 4 * m * case["nsrc"], "flops": 0}
    if op == "spmspv":  # the frontier's rows, and the touched outputs
        e = max(1, nnz * case["nx"] // m)
        out = min(m, e)
        return {"bytes": 16 * case["nx"] + 8 * e + 12 * out, "flops": 2 * e}
    if op == "spgemm":
        # squares of R-MAT fill a large part of the matrix (40M of 268M
        # entries at 2^14 vertices), squares of a lattice about 10 a row
        out = 10 * m if case["graph"] == "lattice" else int(0.15 * m * m * (case["ef"] / 16))
        return {"bytes": csr + 4 * nnz + 4 * m + 8 * out, "flops": 8 * out}
    one = 12 if case["weighted"] else 8
    ne = case["ef"] * m
    return {"bytes": one * ne + 4 * m + 8 * (nnz if case["symmetrize"] else ne), "flops": 0}


# ------------------------------------------------------------------- exact
def _csr64(u, v, w, m):
    """Row ids, columns and float64 values of the symmetric matrix in CSR order."""
    off = u != v
    a, b = u[off].long(), v[off].long()
    key = torch.cat([a * m + b, b * m + a])
    val = torch.cat([w[off], w[off]])
    key, at = key.sort(stable=True)
    first = torch.ones_like(key, dtype=torch.bool)
    first[1:] = key[1:] != key[:-1]
    key, val = key[first], val[at[first]].double()
    return key // m, key % m, val


def _paths64(row, col, val, m, sources):
    """Rounds of relaxation of the rows whose distance went down."""
    ptr = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.bincount(row, minlength=m).cumsum(0)
    out = torch.full((len(sources), m), float("inf"), dtype=torch.float64, device=DEV)
    for dist, s in zip(out, sources):
        dist[s] = 0.0
        live = torch.tensor([s], device=DEV)
        while live.numel():
            start, n = ptr[live], ptr[live + 1] - ptr[live]
            at = torch.repeat_interleave(start - (n.cumsum(0) - n), n)
            e = at + torch.arange(at.numel(), device=DEV)
            d = torch.repeat_interleave(dist[live], n) + val[e]
            to = col[e]
            down = d < dist[to]
            to, d = to[down], d[down]
            dist.scatter_reduce_(0, to, d, "amin")
            live = to.unique()
    unreached = torch.tensor(float(A.SSSP_INF), dtype=torch.float64, device=DEV)
    return torch.where(torch.isinf(out), unreached, out)


def _padded(x, n):
    out = torch.zeros(n, dtype=torch.float64, device=DEV)
    out[:x.numel()] = x
    return out


def exact(case, seed):
    op, m = case["op"], _vertices(case)
    if op not in ("sssp", "sssp_batch", "spgemm", "spmspv", "build"):
        return None  # whole numbers
    u, v, w, gen = _edges(case, seed)
    if op == "sssp":
        s = _connected(u, v, m, 1, gen).tolist()
        return _paths64(*_csr64(u, v, w, m), m, s)[0]
    if op == "sssp_batch":
        s = _connected(u, v, m, case["nsrc"], gen).tolist()
        if len(s) * m > 1 << 24:
            return None  # the rounds of so many sources take too long one by one
        return _paths64(*_csr64(u, v, w, m), m, s)
    if op == "build":
        if w is None:
            w = torch.ones(u.numel(), device=DEV)
        if case["symmetrize"]:
            val = _csr64(u, v, w, m)[2]
        else:
            val = w[u.sort(stable=True).indices].double()
        return {"rowptr": None, "col": None, "val": _padded(val, _room(case)), "nnz": None}
    row, col, val = _csr64(u, v, w, m)
    if op == "spmspv":
        xi, xv, mask = _frontier(case, gen)
        sr = case["semiring"]
        start = 0.0 if sr in (A.SR_PLUS_TIMES, A.SR_BOOL) else float("inf")
        x = torch.full((m,), float("nan"), dtype=torch.float64, device=DEV)
        x[xi.long()] = xv.double()
        use = ~torch.isnan(x[row])
        if mask is not None:
            use &= mask[col] == 0
        xu, a, to = x[row[use]], val[use], col[use]
        hit = to.unique()
        y = torch.zeros(m, dtype=torch.float64, device=DEV)
        if sr == A.SR_PLUS_TIMES:
            y.index_add_(0, to, xu * a)
        elif sr == A.SR_BOOL:
            y[to] = 1.0
        else:
            y.fill_(start if sr == A.SR_MIN_PLUS else -start)
            y.scatter_reduce_(0, to, xu + a if sr == A.SR_MIN_PLUS else xu,
                              "amin" if sr == A.SR_MIN_PLUS else "amax")
        return {"ind": None, "val": _padded(y[hit], m), "count": None}
    # C = A * A, rows of C in blocks that hold their products in memory
    ptr = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.bincount(row, minlength=m).cumsum(0)
    n = ptr[col + 1] - ptr[col]
    done = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    done[1:] = torch.zeros(m, dtype=torch.int64, device=DEV).index_add_(0, row, n).cumsum(0)
    done, ptr_h = done.tolist(), ptr.tolist()
    vals, r0 = [], 0
    while r0 < m:
        r1 = r0 + 1
        while r1 < m and done[r1 + 1] - done[r0] <= 1 << 26:
            r1 += 1
        e0, e1 = ptr_h[r0], ptr_h[r1]
        k = n[e0:e1]
        at = torch.repeat_interleave(ptr[col[e0:e1]] - (k.cumsum(0) - k), k)
        f = at + torch.arange(at.numel(), device=DEV)
        prod = torch.repeat_interleave(val[e0:e1], k) * val[f]
        key = torch.repeat_interleave(row[e0:e1] * m, k) + col[f]
        key, inv = key.unique(return_inverse=True)
        vals.append(torch.zeros(key.numel(), dtype=torch.float64, device=DEV)
                    .index_add_(0, inv, prod))
        r0 = r1
    return {"rowptr": None, "col": None, "val": _padded(torch.cat(vals), _room(case)), "nnz": None}
