"""Graphs with a long run of ids without edges between the others (typed id
blocks): the passes over tiles of edges neither walk the run nor lose the rows
around it."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def blocks(olv, n, m, lo, hi, seed):
    """m uniform edges among the ids outside [lo, hi)."""
    rng = np.random.default_rng(seed)

    def ids(k):
        x = rng.integers(0, n - (hi - lo), k)
        return np.where(x >= lo, x + (hi - lo), x)

    src, dst = np.sort(ids(m)), ids(m)
    rp = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint32)
    return olv.CsrGraph(rp, dst.astype(np.uint32)), src


# runs below and above what a tile walks, at the start and the end, one that
# ends inside a tile of 4096 edges, edges that fill less than one tile
@pytest.mark.parametrize("n,m,lo,hi", [(40_000, 30_000, 10_000, 26_000), (300_000, 20_000, 3_000, 295_000),
                                       (300_000, 20_000, 0, 250_000), (300_000, 20_000, 50_000, 300_000),
                                       (2_000_000, 4_097, 1_000, 1_999_000), (2_000_000, 100, 40, 1_999_960)])
def test_gradient_and_twin(olv, n, m, lo, hi):
    print("empty rows", n, m, lo, hi, flush=True)
    csr, src = blocks(olv, n, m, lo, hi, n + m)
    csr = olv.with_weights_f32_normalized(csr, seed=1)
    rng = np.random.default_rng(0)
    g = olv.Graph(csr)
    B = olv.DeviceBuffer.from_numpy
    w, t = B(csr.weights), B(olv.gen_dirichlet(n, 2))
    r = g.pagerank_weighted(w, t)[0]
    gbar = B(rng.standard_normal(n).astype(np.float32))
    gw, gt, lam = g.pagerank_vjp(w, r, gbar)[:3]
    # grad_w[u -> v] = d r_u lambda_v: one fp32 product after another
    want = np.float32(0.85) * r.numpy()[src] * lam.numpy()[csr.col]
    assert np.allclose(gw.numpy(), want, rtol=3e-7, atol=0)
    s = int(src[0])
    assert np.array_equal(g.bfs(s)[0].numpy(), oracle.bfs(csr.row_ptr, csr.col, s))  # over the renumbered twin


def test_backward_time(olv):
    """A run of 10 M empty rows between the others makes the backward pass take
    longer than one after them by its passes over vectors (1.6 times), not by a
    walk of the run in one workgroup (21 times)."""
    n, m = 12_000_000, 2_000_000
    took = []
    for lo, hi in ((2_000_000, 12_000_000), (1_000_000, 11_000_000)):
        csr, _ = blocks(olv, n, m, lo, hi, 5)
        csr = olv.with_weights_f32_normalized(csr, seed=1)
        g = olv.Graph(csr)
        B = olv.DeviceBuffer.from_numpy
        w, r, gbar = B(csr.weights), B(np.full(n, 1 / n, np.float32)), B(np.ones(n, np.float32))
        took.append(min(g.pagerank_vjp(w, r, gbar)[3].elapsed_ms for _ in range(6)))
        g.close()
    print("backward after / between", took, flush=True)
    assert took[1] < 4 * took[0]
