"""Buffers that a graph lends to its calls: two calls in flight at once, as from
several threads on a graph whose plans are already built, never hold the same ones.
Building those plans is left to one thread."""
import threading

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def test_calls_share_a_graph(olv):
    rng = np.random.default_rng(3)
    n, m = 3001, 20000
    src, dst = np.sort(rng.integers(0, n, m)), rng.integers(0, n, m)
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint32)
    csr = olv.CsrGraph(rp, dst.astype(np.uint32), rng.integers(1, 65, m).astype(np.int32))
    g = olv.Graph(csr, transpose=True)
    srcs = rng.integers(0, n, (4, 40)).astype(np.uint32)
    levels = [np.stack([oracle.bfs(rp, csr.col, int(s)) for s in row]) for row in srcs]
    dist = [oracle.dijkstra(rp, csr.col, csr.weights, int(row[0])) for row in srcs]
    g.bfs_batched(srcs[0]), g.sssp(int(srcs[0][0]))  # what the graph keeps for good is built here
    bad = []

    def run(i):
        for r in range(5):
            k = 40 - 17 * (r % 2)  # the kept buffers' size changes hands too
            if not np.array_equal(g.bfs_batched(srcs[i][:k])[0].numpy().reshape(k, n), levels[i][:k]):
                bad.append(("bfs", i, r))
            if not np.array_equal(g.sssp(int(srcs[i][0]))[0].numpy(), dist[i]):
                bad.append(("sssp", i, r))

    print("threads on one graph", flush=True)
    ts = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
