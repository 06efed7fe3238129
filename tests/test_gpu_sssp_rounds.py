"""SSSP by direct relaxation where its layout changes: vertex counts that do
not fill the last word of mark bytes, hub rows cut into items, and both sides
of the sizes up to which relaxations lower candidate copies instead of the
distances.  Distances are whole numbers: equal to Dijkstra's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def graph(olv, n, m, hub, seed):
    """m uniform edges plus `hub` out-edges of vertex n // 2, weights 1..64."""
    rng = np.random.default_rng(seed)
    src = np.concatenate([rng.integers(0, n, m), np.full(hub, n // 2)])
    dst = rng.integers(0, n, src.size)
    o = np.lexsort((dst, src))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, src + 1, 1)
    return olv.CsrGraph(np.cumsum(rp).astype(np.uint32), dst[o].astype(np.uint32),
                        rng.integers(1, 65, src.size).astype(np.int32))


@pytest.mark.parametrize("n,m,hub", [(1, 2, 0), (2, 3, 0), (3, 7, 0), (5, 20, 1500), (1023, 4000, 1024),
                                     (4097, 20000, 5000), ((1 << 20), 1 << 21, 3000), ((1 << 20) + 3, 1 << 21, 3000),
                                     (600_000, 1_500_000, 0), (600_001, 1_500_000, 0)])
def test_direct_rounds(olv, n, m, hub):
    print("sssp rounds", n, m, hub, flush=True)
    csr = graph(olv, n, m, hub, n)
    g = olv.Graph(csr, transpose=False)
    for s in {0, n // 2, n - 1}:
        ref = oracle.dijkstra(csr.row_ptr, csr.col, csr.weights, s)
        assert np.array_equal(g.sssp(s)[0].numpy(), ref), s


def test_batched_rounds(olv):
    # three instances of an odd graph: instance boundaries inside a mark word
    csr = graph(olv, 333, 2000, 1100, 1)
    g = olv.Graph(csr, transpose=False)
    srcs = np.array([5, 166, 332], np.uint32)
    out = g.sssp_batched(srcs)[0].numpy().reshape(3, -1)
    for i, s in enumerate(srcs):
        assert np.array_equal(out[i], oracle.dijkstra(csr.row_ptr, csr.col, csr.weights, int(s))), s


def test_frontiers_larger_than_a_workgroup_holds(olv):
    """Nine million vertices, all improved in the first round: compacting
    workgroups take several runs of vertices and hand their share of the queue
    on more than once.  With unit weights the distances are BFS levels."""
    n = 9_000_003
    rng = np.random.default_rng(2)
    src = np.concatenate([np.zeros(n - 1, np.int64), rng.integers(0, n, 2_000_000)])
    dst = np.concatenate([np.arange(1, n), rng.integers(0, n, 2_000_000)])
    o = np.argsort(src, kind="stable")
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint32)
    csr = olv.CsrGraph(rp, dst[o].astype(np.uint32), np.ones(src.size, np.int32))
    print("sssp rounds, wide frontier", flush=True)
    g = olv.Graph(csr, transpose=False)
    for s in (0, int(src[-1])):
        assert np.array_equal(g.sssp(s)[0].numpy(), oracle.bfs(rp, csr.col, s)), s


def test_more_vertices_than_the_bins_take(olv):
    n, m = (1 << 24) + 5, 1 << 25
    rng = np.random.default_rng(9)
    src = np.sort(rng.integers(0, n, m, dtype=np.int64))
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint32)
    csr = olv.CsrGraph(rp, rng.integers(0, n, m).astype(np.uint32), np.ones(m, np.int32))
    print("sssp rounds, 2^24 + 5 vertices", flush=True)
    s = int(src[m // 2])
    ref = oracle.bfs(rp, csr.col, s)
    assert (ref < 0x7FFFFFFF).sum() > n // 2
    assert np.array_equal(olv.Graph(csr, transpose=False).sssp(s)[0].numpy(), ref)
