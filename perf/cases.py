"""The timed cases: what programs have this library do, over the sizes they do
it at.

Every graph is made on the GPU from a seed and handed to the library as an edge
list (``olv_graph_from_coo``), as a program whose edges already sit in device
memory does; the calls go through the C ABI (``include/olive_hip.h``) with
torch tensors as inputs and outputs, or through ``olive_amd.autograd``.

A case is ``{"op": ..., "graph": ..., sizes}``:

op        bfs            levels from one source (``olv_bfs``)
          bfs_batched    levels from k sources in one sweep (``olv_bfs_batched``)
          sssp           distances over int32 weights (``olv_sssp``)
          pagerank       ``iters`` fp32 iterations (``olv_pagerank_f32``)
          train          differentiable PageRank: forward fixed point and the
                         gradients of weights and teleport vector
          tangent        the same fixed point in forward mode (a dual number
                         through ``torch.autograd.forward_ad``)
          ingest         edge-list text in device memory to a resident graph
                         with both CSRs (``olv_graph_from_edge_list_text``)
graph     rmat           skewed degrees, RMAT (0.57, 0.19, 0.19, 0.05) ids
                         folded to n vertices, m edges
          uniform        m edges with uniform endpoints
          grid           rows x cols, edges to the four neighbours
"""
import ctypes
import math

import numpy as np
import torch
from torch.autograd import forward_ad

import olive_amd
from olive_amd import autograd
from olive_amd._lib import OLV_BUILD_TRANSPOSE, OLV_W_I32, OLV_W_NONE, check, lib

INF = olive_amd.INF
DAMPING = 0.85
TOL = 1e-6
RMAT = (0.57, 0.19, 0.19)


# ------------------------------------------------------------------- cases
def listed():
    return [
        # One traversal of a small mesh (the repository's 128 x 128 grid): 255
        # levels of at most 128 vertices, the call whose cost is latency alone.
        {"name": "bfs_grid_128x128", "op": "bfs", "graph": "grid", "rows": 128, "cols": 128},
        # A mesh of a quarter million vertices with ragged sides: many levels,
        # each far too small for the chip (road networks, image grids).
        {"name": "bfs_grid_601x389", "op": "bfs", "graph": "grid", "rows": 601, "cols": 389},
        # The benchmark's traversal: a social-network graph of 4.2 M vertices
        # and 67 M edges from one source.
        {"name": "bfs_rmat_22", "op": "bfs", "graph": "rmat", "n": 1 << 22, "m": 1 << 26},
        # Many sources of one graph at once (landmarks, closeness): 256 sources
        # on RMAT-20, called without a plan.
        {"name": "bfs_256_rmat_20", "op": "bfs_batched", "graph": "rmat", "n": 1 << 20, "m": 1 << 24, "k": 256},
        # Shortest paths on a skewed graph (hub vertices) of ordinary, odd size.
        {"name": "sssp_rmat_250k", "op": "sssp", "graph": "rmat", "n": 250007, "m": 4000037},
        # The benchmark's shortest paths: uniform graph, 4.2 M vertices, 33.6 M
        # edges, weights 1..64.
        {"name": "sssp_uniform_4m", "op": "sssp", "graph": "uniform", "n": 1 << 22, "m": 1 << 25},
        # The smallest ranking call: 20 iterations over 4096 vertices.
        {"name": "pagerank_rmat_12", "op": "pagerank", "graph": "rmat", "n": 1 << 12, "m": 1 << 16, "iters": 20},
        # The benchmark's ranking: RMAT-20, 20 iterations.
        {"name": "pagerank_rmat_20", "op": "pagerank", "graph": "rmat", "n": 1 << 20, "m": 1 << 24, "iters": 20},
        # Ranking a graph without hubs (no locality to find), odd sizes.
        {"name": "pagerank_uniform_700k", "op": "pagerank", "graph": "uniform", "n": 700001, "m": 9000011,
         "iters": 20},
        # A training step through the fixed point: the weights come from an
        # upstream operation (a new tensor each step), forward and backward.
        {"name": "train_rmat_20", "op": "train", "graph": "rmat", "n": 1 << 20, "m": 1 << 24},
        # A directional derivative on a small graph (forward mode).
        {"name": "tangent_rmat_16", "op": "tangent", "graph": "rmat", "n": 1 << 16, "m": 1 << 20},
        # Edge-list text of 8.4 M edges to CSR and in-CSR.
        {"name": "ingest_rmat_19", "op": "ingest", "graph": "rmat", "n": 1 << 19, "m": 1 << 23},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["bfs", "bfs", "bfs_batched", "sssp", "sssp", "pagerank", "pagerank", "train", "tangent", "ingest"])
    if op == "bfs" and rng.random() < 0.4:
        return {"op": op, "graph": "grid", "rows": _log_uniform(rng, 16, 600), "cols": _log_uniform(rng, 16, 390)}
    # edges per vertex as in the listed graphs, from sparse to twice the usual
    ranges = {
        "bfs": (1 << 10, 1 << 26), "bfs_batched": (1 << 12, 1 << 24), "sssp": (1 << 12, 1 << 25),
        "pagerank": (1 << 12, 1 << 24), "train": (1 << 12, 1 << 24), "tangent": (1 << 12, 1 << 22),
        "ingest": (1 << 10, 1 << 23),
    }
    m = _log_uniform(rng, *ranges[op])
    n = max(64, int(m / rng.uniform(6.0, 32.0)))
    case = {"op": op, "graph": rng.choice(["rmat", "rmat", "uniform"]), "n": n, "m": m}
    if op == "bfs_batched":
        case["k"] = rng.choice([5, 32, 64, 100, 256])
    if op == "pagerank":
        case["iters"] = rng.choice([10, 20, 30])
    return case


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed + 1) + 17)
    return g


def _grid_edges(rows, cols):
    v = torch.arange(rows * cols, device="cuda", dtype=torch.int64).view(rows, cols)
    pairs = [(v[:-1], v[1:]), (v[1:], v[:-1]), (v[:, :-1], v[:, 1:]), (v[:, 1:], v[:, :-1])]
    src = torch.cat([a.reshape(-1) for a, _ in pairs])
    dst = torch.cat([b.reshape(-1) for _, b in pairs])
    return src.to(torch.int32), dst.to(torch.int32)


def _rmat_edges(n, m, gen):
    a, b, c = RMAT
    src = torch.zeros(m, device="cuda", dtype=torch.int32)
    dst = torch.zeros(m, device="cuda", dtype=torch.int32)
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(m, device="cuda", generator=gen)
        down = r >= a + b
        right = ((r >= a) & ~down) | (r >= a + b + c)
        src.mul_(2).add_(down)
        dst.mul_(2).add_(right)
    return src % n, dst % n


def _edges(case, gen):
    """(n, src, dst): int32 device arrays, edges in no particular order."""
    if case["graph"] == "grid":
        src, dst = _grid_edges(case["rows"], case["cols"])
        return case["rows"] * case["cols"], src, dst
    n, m = case["n"], case["m"]
    if case["graph"] == "rmat":
        return (n,) + _rmat_edges(n, m, gen)
    src = torch.randint(0, n, (m,), device="cuda", dtype=torch.int32, generator=gen)
    dst = torch.randint(0, n, (m,), device="cuda", dtype=torch.int32, generator=gen)
    return n, src, dst


def _sorted_by_source(src, dst):
    order = torch.argsort(src, stable=True)
    return src[order], dst[order]


def _source(src, n, gen, k=1):
    """k vertices that have out-edges, uniformly."""
    has = torch.zeros(n, device="cuda", dtype=torch.bool)
    has[src.long()] = True
    ids = has.nonzero().view(-1)
    pick = torch.randint(0, ids.numel(), (k,), device="cuda", generator=gen)
    return ids[pick].to(torch.int32).cpu().numpy().view(np.uint32)


def _stochastic_weights(src, n, gen):
    """fp32 edge weights that sum to 1 over each source (whole numbers until
    the division, so the same seed gives the same bits)."""
    x = torch.randint(1, 1025, (src.numel(),), device="cuda", generator=gen)
    total = torch.zeros(n, device="cuda", dtype=torch.int64).index_add_(0, src.long(), x)
    return (x.double() / total[src.long()].double()).float()


def _unit_vector(n, gen):
    """A probability vector (exact up to one fp32 rounding per entry)."""
    x = torch.randint(1, 1025, (n,), device="cuda", generator=gen)
    return (x.double() / x.sum().double()).float()


def _scale(seed):
    """What the upstream operation multiplies the weights by (exact in binary)."""
    return 0.96875 + 0.03125 * (seed % 2)


def _signed(n, gen):
    return torch.randint(-1024, 1025, (n,), device="cuda", generator=gen).float() / 1024.0


def _edge_list_text(n, src, dst):
    """The edge list as text in device memory: header "n m", "src dst" lines."""
    def digits(x):
        d = torch.ones_like(x)
        for p in range(1, 10):
            d += x >= 10 ** p
        return d

    header = torch.tensor(list(("%d %d\n" % (n, src.numel())).encode()), dtype=torch.uint8, device="cuda")
    cols = [src.long(), dst.long()]
    width = [digits(c) for c in cols]
    end = torch.cumsum(width[0] + width[1] + 2, 0) + header.numel()
    pos = end - (width[0] + width[1] + 2)
    text = torch.empty(int(end[-1]) if end.numel() else header.numel(), dtype=torch.uint8, device="cuda")
    text[:header.numel()] = header
    for c, w, sep in ((cols[0], width[0], " "), (cols[1], width[1], "\n")):
        for k in range(int(w.max())):
            at = w > k
            text[(pos + w - 1 - k)[at]] = (48 + (c[at] // 10 ** k) % 10).to(torch.uint8)
        pos = pos + w
        text[pos] = ord(sep)
        pos = pos + 1
    return text


class Handle:
    """A resident graph (olv_graph) of edges in device memory."""

    def __init__(self, n, src, dst, weights=None):
        olive_amd.init()
        self.n, self.m = n, src.numel()
        h = ctypes.c_void_p()
        torch.cuda.current_stream().synchronize()
        check(lib().olv_graph_from_coo(ctypes.byref(h), n, self.m, src.data_ptr(), dst.data_ptr(),
                                       None if weights is None else weights.data_ptr(),
                                       OLV_W_NONE if weights is None else OLV_W_I32, OLV_BUILD_TRANSPOSE, None),
              "olv_graph_from_coo")
        self.h = h

    def __del__(self):
        if getattr(self, "h", None) and lib is not None:  # (None while the interpreter ends)
            lib().olv_graph_destroy(self.h)
            self.h = None


def prepare(case, seed):
    gen = _generator(seed)
    n, src, dst = _edges(case, gen)
    op = case["op"]
    if op == "ingest":
        olive_amd.init()
        return {"case": case, "text": _edge_list_text(n, src, dst), "n": n, "m": src.numel()}
    if op in ("train", "tangent"):
        src, dst = _sorted_by_source(src, dst)  # the weights' order is the CSR's
    weights = None
    if op == "sssp":
        weights = torch.randint(1, 65, (src.numel(),), device="cuda", dtype=torch.int32, generator=gen)
    st = {"case": case, "g": Handle(n, src, dst, weights)}
    if op == "bfs" or op == "sssp":
        st["source"] = int(_source(src, n, gen)[0])
        st["out"] = torch.empty(n, device="cuda", dtype=torch.int32)
    elif op == "bfs_batched":
        st["sources"] = np.ascontiguousarray(_source(src, n, gen, case["k"]))
        st["out"] = torch.empty((case["k"], n), device="cuda", dtype=torch.int32)
    elif op == "pagerank":
        st["out"] = torch.empty(n, device="cuda", dtype=torch.float32)
    else:
        st["w"] = _stochastic_weights(src, n, gen)
        st["scale"] = torch.tensor(_scale(seed), device="cuda")
        st["t"] = _unit_vector(n, gen)
        if op == "train":
            st["cotangent"] = _signed(n, gen)
        else:
            st["dw"] = _signed(src.numel(), gen) * st["w"]
            st["dt"] = _signed(n, gen) * st["t"]
    return st


# --------------------------------------------------------------------- run
def _out_arrays(h, n, m):
    """Copies of a graph's resident arrays as torch tensors."""
    ptr = [ctypes.c_void_p() for _ in range(6)]
    check(lib().olv_graph_device_arrays(h, *[ctypes.byref(p) for p in ptr]), "olv_graph_device_arrays")
    out = []
    for p, count in ((ptr[0], n + 1), (ptr[1], m), (ptr[3], n + 1), (ptr[4], m), (ptr[5], m)):
        x = torch.empty(count, device="cuda", dtype=torch.int32)
        check(lib().olv_memcpy_d2d(x.data_ptr(), p, count * 4), "olv_memcpy_d2d")
        out.append(x)
    return out


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "ingest":
        h = ctypes.c_void_p()
        check(lib().olv_graph_from_edge_list_text(ctypes.byref(h), ctypes.c_char_p(st["text"].data_ptr()),
                                                  st["text"].numel(), OLV_BUILD_TRANSPOSE, None),
              "olv_graph_from_edge_list_text")
        out = _out_arrays(h, st["n"], st["m"])
        check(lib().olv_graph_destroy(h), "olv_graph_destroy")
        return out
    g = st["g"]
    if op == "bfs":
        check(lib().olv_bfs(g.h, st["source"], st["out"].data_ptr(), 0, None), "olv_bfs")
        return st["out"]
    if op == "bfs_batched":
        check(lib().olv_bfs_batched(g.h, st["sources"].ctypes.data, case["k"], st["out"].data_ptr(), 0, None),
              "olv_bfs_batched")
        return st["out"]
    if op == "sssp":
        check(lib().olv_sssp(g.h, st["source"], None, st["out"].data_ptr(), 0, None), "olv_sssp")
        return st["out"]
    if op == "pagerank":
        check(lib().olv_pagerank_f32(g.h, DAMPING, case["iters"], 0.0, st["out"].data_ptr(), 0, None),
              "olv_pagerank_f32")
        return st["out"]
    w = st["w"] * st["scale"]
    if op == "train":
        w.requires_grad_(True)
        t = st["t"].detach().requires_grad_(True)
        r = autograd.pagerank(g, w, t, damping=DAMPING, tol=TOL)
        gw, gt = torch.autograd.grad(r, [w, t], st["cotangent"])
        return {"r": r.detach(), "grad_w": gw, "grad_t": gt}
    with forward_ad.dual_level():
        wd = forward_ad.make_dual(w, st["dw"])
        td = forward_ad.make_dual(st["t"], st["dt"])
        r = autograd.pagerank(g, wd, td, damping=DAMPING, tol=TOL)
        primal, tangent = forward_ad.unpack_dual(r)
        return {"r": primal.detach(), "dr": tangent.detach()}


# -------------------------------------------------------------------- work
def _sizes(case):
    if case["graph"] == "grid":
        r, c = case["rows"], case["cols"]
        return r * c, 4 * r * c - 2 * r - 2 * c
    return case["n"], case["m"]


def work(case):
    """Bytes and operations that a pass needs at the least: the graph read
    once for a traversal, once per iteration for a fixed point whose every
    iteration needs the one before."""
    n, m = _sizes(case)
    op = case["op"]
    if op == "bfs":
        return {"bytes": 4 * m + 4 * (n + 1) + 4 * n, "flops": 0}
    if op == "bfs_batched":
        return {"bytes": 4 * m + 4 * (n + 1) + 4 * n * case["k"], "flops": 0}
    if op == "sssp":
        return {"bytes": 8 * m + 4 * (n + 1) + 4 * n, "flops": m}
    if op == "pagerank":
        return {"bytes": case["iters"] * (4 * m + 12 * n), "flops": case["iters"] * (m + 4 * n)}
    if op in ("train", "tangent"):
        # index and weight of every edge per iteration, two solves of about
        # log(tol) / log(damping) iterations; weights read and (train) their
        # gradient written once more
        it = 2 * 40
        return {"bytes": it * (8 * m + 12 * n) + 8 * m, "flops": it * (2 * m + 4 * n)}
    digits = 2 * len(str(n)) + 2
    return {"bytes": digits * m + 12 * m + 8 * (n + 1), "flops": 0}


# ------------------------------------------------------------------- exact
class _RowSums:
    """sums(x)[v] = sum of x over the edges whose row is v, in 64 bits (a
    running sum over the edges in row order, so hub rows cost no more)."""

    def __init__(self, rows, n):
        self.order = torch.argsort(rows, stable=True)
        self.end = torch.cumsum(torch.bincount(rows, minlength=n), 0)

    def __call__(self, x):
        run = torch.cat([x.new_zeros(1), torch.cumsum(x[self.order], 0)])[self.end]
        return torch.diff(run, prepend=run.new_zeros(1))


def _solve(sums, cols, w, base, start, stop):
    """x = base + d * A x in 64 bits, A x = sums(w * x[cols]), from `start` to
    an L1 change below `stop`."""
    d, x = float(np.float32(DAMPING)), start
    while True:
        nx = base + d * sums(w * x[cols])
        change = float((nx - x).abs().sum())
        x = nx
        if change < stop:
            return x


def exact(case, seed):
    op = case["op"]
    if op not in ("pagerank", "train", "tangent"):
        return None  # whole numbers
    gen = _generator(seed)
    n, src, dst = _edges(case, gen)
    d = float(np.float32(DAMPING))
    if op == "pagerank":
        src, dst = src.long(), dst.long()
        deg = torch.bincount(src, minlength=n).double()
        inv = torch.where(deg > 0, 1.0 / deg.clamp(min=1), torch.zeros_like(deg))
        r = torch.full((n,), 1.0 / n, device="cuda", dtype=torch.float64)
        sums = _RowSums(dst, n)
        for _ in range(case["iters"]):
            r = d * sums((r * inv)[src]) + (1.0 - d) / n
        return r
    src, dst = _sorted_by_source(src, dst)
    w = _stochastic_weights(src, n, gen)
    t = _unit_vector(n, gen)
    if op == "train":
        c = _signed(n, gen).double()
    else:
        dw, dt = (_signed(src.numel(), gen) * w).double(), (_signed(n, gen) * t).double()
    w = w * _scale(seed)
    src, dst, w, t = src.long(), dst.long(), w.double(), t.double()
    keep = float(np.float32(1.0) - np.float32(DAMPING))
    into = _RowSums(dst, n)
    r = _solve(into, src, w, keep * t, t, TOL)
    if op == "train":
        lam = _solve(_RowSums(src, n), dst, w, c, c, TOL * float(c.abs().sum()))
        return {"r": r, "grad_w": d * r[src] * lam[dst], "grad_t": keep * lam}
    s = d * into(dw * r[src]) + keep * dt
    return {"r": r, "dr": _solve(into, src, w, s, s / keep, TOL)}
