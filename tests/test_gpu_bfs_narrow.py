"""BFS levels run in one workgroup: frontiers on both sides of the sizes that
fit it, hubs among them, paths longer than one launch may run, and the hand-over
to the expansion kernels and back.  Levels are equal to the oracle's."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def layered(olv, widths, extra, seed):
    """Layer i + 1's vertices each hang on a vertex of layer i, which they point
    back to; `extra` edges join vertices of one layer.  Ids are shuffled."""
    rng = np.random.default_rng(seed)
    off = np.concatenate([[0], np.cumsum(widths)])
    n = int(off[-1])
    layer = np.repeat(np.arange(len(widths)), widths)
    child = np.arange(widths[0], n)
    lp = layer[child] - 1
    parent = off[lp] + rng.integers(0, np.asarray(widths)[lp])
    a = rng.integers(0, n, extra)
    b = off[layer[a]] + rng.integers(0, np.asarray(widths)[layer[a]])
    perm = rng.permutation(n)
    src, dst = perm[np.concatenate([parent, child, a])], perm[np.concatenate([child, parent, b])]
    o = np.lexsort((dst, src))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, src + 1, 1)
    return olv.CsrGraph(np.cumsum(rp).astype(np.uint32), dst[o].astype(np.uint32)), int(perm[0])


CASES = {
    "path": ([1] * 20000, 0),
    "narrow": ([1, 2, 63, 64, 65, 500, 1023, 1024, 1025, 700] * 4, 9000),
    "queue_limit": ([1, 40, 2047, 30, 2048, 1, 2049, 7, 2050, 5, 5000, 1, 300, 6000, 100] + [3] * 40, 2000),
    "edge_limit": ([1, 1365, 1366, 1364, 700, 2000, 1900, 1, 800] * 2, 30000),
    "hubs": ([1] * 20 + [3000, 1, 5000, 2, 1, 9000] + [1] * 30 + [4097, 4096, 4095, 1] + [2] * 50, 3000),
    "deep_again": (([1] * 40 + [7000]) * 3, 0),
}


@pytest.mark.parametrize("name", CASES)
def test_narrow_levels(olv, name):
    from olive_amd import _lib

    csr, src = layered(olv, *CASES[name], seed=len(name))
    ref = oracle.bfs(csr.row_ptr, csr.col, src)
    assert csr.n > 16384  # not a graph for the small-graph kernel
    for flags in (0, _lib.OLV_GRAPH_ORDER, _lib.OLV_NO_DIRECTION_OPT):
        g = olv.Graph(csr, transpose=True)
        for run in range(3):  # the first run starts with launch pairs, later ones with what it learned
            print("bfs narrow", name, flags, run, flush=True)
            lv, st = g.bfs(src, flags=flags)
            assert np.array_equal(lv.numpy(), ref), (flags, run)
            assert st.iterations == ref.max() + 1
            if flags == _lib.OLV_NO_DIRECTION_OPT:
                assert st.edges_inspected == csr.m
        lv = olv.DeviceBuffer(csr.n, np.int32)
        _lib.check(_lib.lib().olv_bfs_noalloc(g.h, src, lv.c, flags | _lib.OLV_NO_DIRECTION_OPT, None), "noalloc")
        assert np.array_equal(lv.numpy(), ref), flags
        seeds = np.flatnonzero(ref % 97 == 5)[:300].astype(np.uint32)
        if seeds.size:
            want = np.min([oracle.bfs(csr.row_ptr, csr.col, int(s)) for s in seeds[:40]], axis=0)
            assert np.array_equal(g.bfs_multisource(seeds[:40], flags=flags)[0].numpy(), want), flags
        plan = ctypes.c_void_p()
        s1 = np.array([src], np.uint32)
        _lib.check(_lib.lib().olv_plan_bfs(g.h, s1.ctypes.data, 1, lv.c, flags, ctypes.byref(plan)), "plan")
        for _ in range(3):
            _lib.check(_lib.lib().olv_plan_launch(plan, None), "launch")
            assert np.array_equal(lv.numpy(), ref), flags
        _lib.lib().olv_plan_destroy(plan)


@pytest.mark.parametrize("extra", [0, 9000, 40000])  # mean degrees 2, 4 and 8: lanes per row 2, 4 and 8
def test_small_graph_levels(olv, extra):
    widths = [1, 3, 127, 128, 129, 255, 256, 257, 60, 511, 512, 513, 1023, 1024, 1025, 40, 64, 63, 65]
    csr, src = layered(olv, widths, extra, seed=extra + 1)
    assert csr.n <= 16384 and np.diff(csr.row_ptr.astype(np.int64)).max() <= 256  # for the small-graph kernel
    ref = oracle.bfs(csr.row_ptr, csr.col, src)
    g = olv.Graph(csr, transpose=False)
    print("bfs small", extra, flush=True)
    lv, st = g.bfs(src)
    assert np.array_equal(lv.numpy(), ref)
    assert (st.iterations, st.edges_inspected, st.vertices_reached) == (ref.max() + 1, csr.m, csr.n)
    seeds = np.flatnonzero(ref == 5).astype(np.uint32)
    want = np.min([oracle.bfs(csr.row_ptr, csr.col, int(s)) for s in seeds[:9]], axis=0)
    assert np.array_equal(g.bfs_multisource(seeds[:9])[0].numpy(), want)


@pytest.mark.parametrize("name", ["narrow", "queue_limit", "edge_limit", "hubs"])
def test_narrow_levels_many_vertices(olv, name):
    # more vertices than the bitmap in LDS holds: isolated ones between the others
    from olive_amd import _lib

    small, src = layered(olv, *CASES[name], seed=len(name))
    step = 800_000 // small.n + 1
    deg = np.zeros(small.n * step, np.int64)
    deg[::step] = np.diff(small.row_ptr.astype(np.int64))
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    csr = olv.CsrGraph(rp, small.col * np.uint32(step))
    ref = oracle.bfs(csr.row_ptr, csr.col, src * step)
    for flags in (0, _lib.OLV_GRAPH_ORDER, _lib.OLV_NO_DIRECTION_OPT):
        g = olv.Graph(csr, transpose=True)
        for run in range(3):
            print("bfs narrow, many vertices", name, flags, run, flush=True)
            lv, st = g.bfs(src * step, flags=flags)
            assert np.array_equal(lv.numpy(), ref), (flags, run)
            assert st.iterations == ref[ref < 0x7FFFFFFF].max() + 1
