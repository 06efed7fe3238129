"""Batched BFS pull levels where a wave records its one-lane rows together: more
such rows than the rule asks for, with rows of every other width beside them."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [32, 33, 96, 255, 256, 300])  # 32: one lane a row still
def test_wide_rows(olv, k):
    n = 420_003
    rng = np.random.default_rng(k)
    deg = np.zeros(n, np.int64)
    deg[rng.choice(n, 340_000, replace=False)] = 3  # in-degrees: one lane, eight, a wave, a workgroup, pieces
    deg[rng.choice(n, 300, replace=False)] = np.repeat([9, 40, 100, 700, 3000, 20_000], 50)
    dst = np.repeat(np.arange(n), deg)
    src = rng.integers(0, n, dst.size)
    o = np.lexsort((dst, src))
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint32)
    csr = olv.CsrGraph(rp, dst[o].astype(np.uint32))
    g = olv.Graph(csr, transpose=True)
    srcs = rng.integers(0, n, k).astype(np.uint32)
    print("batched bfs wide rows", k, flush=True)
    lv, st = g.bfs_batched(srcs)
    assert st.bottom_up_levels > 0
    assert oracle.bfs_verify(csr.row_ptr, csr.col, srcs, lv.numpy().reshape(k, n)) == -1
