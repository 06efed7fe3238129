"""The source-segmented pull plan, built on the device: row pieces at the
edges of every capacity class, cut pieces, partial segments, rows of every
combine tier, and graphs on both sides of the line below which the plan has
no segment pass.

Tolerances, as for the other PageRank tests: 1e-5 maximum relative error
against the fp64 oracle; the weighted solves against the per-row pull over
the same numbering (same terms, another order) 1e-5 relative L2 for ranks and
1e-4 for gradients and tangents.
"""
import numpy as np
import pytest

import oracle
from olive_amd import _lib

pytestmark = pytest.mark.gpu

# entries of a (row, segment) piece around each capacity and each cut
LENGTHS = [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 24, 25, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 192, 193, 256, 257, 384,
           385, 512, 513, 768, 769, 1024, 1025, 1536, 1537, 2049]
# terms of a row around the combine's tiers
TERMS = [15, 16, 17, 127, 128, 129, 1023, 1024, 1025, 4097, 16384]


def edges_csr(olv, n, src, dst, w=None):
    order = np.lexsort((dst, src))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, np.asarray(src) + 1, 1)
    return olv.CsrGraph(np.cumsum(rp).astype(np.uint32), np.asarray(dst)[order].astype(np.uint32), w)


def ladder(olv, n, fill, hub, seed):
    """Row k's in-list: LENGTHS[k] consecutive sources at a random place (so
    one or two segments), rows of TERMS scattered sources, one of `hub`, and
    `fill` uniform edges into the remaining rows."""
    rng = np.random.default_rng(seed)
    src, dst = [], []
    v = 0
    for ln in LENGTHS * 3:
        s0 = int(rng.integers(0, max(1, n - ln)))
        src.append(np.arange(s0, s0 + ln) % n)
        dst.append(np.full(ln, v))
        v += 1
    for ln in TERMS + [hub]:
        src.append(rng.choice(n, size=min(ln, n), replace=False))
        dst.append(np.full(src[-1].size, v))
        v += 1
    src.append(rng.integers(0, n, fill))
    dst.append(rng.integers(v, n, fill))
    return edges_csr(olv, n, np.concatenate(src), np.concatenate(dst))


CASES = {
    # name: (vertices, uniform edges, hub row) -- 3 segments and 1695 sources of
    # a fourth; one segment exactly; one vertex past it; no segment pass;
    # few edges but a row too long for the single launch
    "segmented": (100003, 600000, 50000),
    "one_segment": (32768, 520000, 20000),
    "segment_plus_one": (32769, 520000, 20000),
    "segment_plus_six": (32774, 520000, 20000),
    "single_launch": (100003, 300000, 16384),
    "few_edges_long_row": (100003, 1000, 70000),
    # lanes with four short rows and more: groups of them of at most two, at
    # most four and more terms
    "many_short_rows": (2200003, 3000000, 50000),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_plain_against_oracle(olv, name):
    print("pull plan", name, flush=True)
    n, fill, hub = CASES[name]
    csr = ladder(olv, n, fill, hub, 3)
    g = olv.Graph(csr)
    ref, _, _ = oracle.pagerank(csr.row_ptr, csr.col, 7, epsilon=0.0)
    a = g.pagerank(7, epsilon=0.0)[0].numpy()
    assert float(np.max(np.abs(a - ref) / ref)) <= 1e-5
    assert np.array_equal(a, g.pagerank(7, epsilon=0.0)[0].numpy())  # fixed order: the same bits


@pytest.mark.parametrize("name", sorted(CASES))
def test_weighted_against_row_pull(olv, name):
    print("pull plan weighted", name, flush=True)
    n, fill, hub = CASES[name]
    rng = np.random.default_rng(5)
    csr = olv.with_weights_f32_normalized(ladder(olv, n, fill, hub, 4), seed=2)
    g = olv.Graph(csr)
    B = olv.DeviceBuffer.from_numpy
    w, t = B(csr.weights), B(olv.gen_dirichlet(n, 7))
    gbar = B(rng.standard_normal(n).astype(np.float32))
    # a tangent of about the ranks' L1 size: its solve stops on an absolute change
    dt = B((rng.standard_normal(n) / n).astype(np.float32))
    dw = B((rng.standard_normal(csr.m) * 1e-3).astype(np.float32))

    def rel(x, y):
        x, y = x.numpy().astype(np.float64), y.numpy().astype(np.float64)
        return np.linalg.norm(x - y) / np.linalg.norm(y)

    r0 = g.pagerank_weighted(w, t, flags=_lib.OLV_PR_ROW_PULL)[0]
    r1 = g.pagerank_weighted(w, t)[0]
    assert rel(r1, r0) <= 1e-5
    for x, y in zip(g.pagerank_vjp(w, r0, gbar)[:3], g.pagerank_vjp(w, r0, gbar, flags=_lib.OLV_PR_ROW_PULL)[:3]):
        assert rel(x, y) <= 1e-4
    j0 = g.pagerank_jvp(w, r0, dw, dt, flags=_lib.OLV_PR_ROW_PULL)[0]
    assert rel(g.pagerank_jvp(w, r0, dw, dt)[0], j0) <= 1e-4


@pytest.mark.parametrize("name", ["segmented", "single_launch"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_not_finite_stays_in_its_rows(olv, name, bad):
    """Weights and teleports that are not finite reach the rows that the per-row
    pull says and no others, whatever pieces share a task with theirs."""
    print("pull plan not finite", name, bad, flush=True)
    n, fill, hub = CASES[name]
    csr = olv.with_weights_f32_normalized(ladder(olv, n, fill, hub, 4), seed=2)
    rng = np.random.default_rng(8)
    w, t = csr.weights.copy(), olv.gen_dirichlet(n, 7)
    w[rng.integers(0, csr.m, 12)] = bad
    t[rng.integers(0, n, 3)] = bad
    g = olv.Graph(csr)
    B = olv.DeviceBuffer.from_numpy
    dw, dt = B(w), B(t)
    for iters in (1, 2):
        out = []
        for flags in (0, _lib.OLV_PR_ROW_PULL):
            r = olv.DeviceBuffer(n, np.float32)
            rc = _lib.lib().olv_pagerank_weighted_f32(g.h, dw.c, dt.c, 0.85, 1e-6, iters, r.c, flags, None)
            assert rc == _lib.OLV_ENOCONV
            out.append(r.numpy())
        a, b = out
        assert np.array_equal(np.isnan(a), np.isnan(b)) and not np.isfinite(a).all()
        fin = np.isfinite(b)
        assert fin.sum() > n // 4  # the rows that nothing of it reaches
        assert np.array_equal(a[~fin], b[~fin], equal_nan=True)
        assert np.linalg.norm(a[fin].astype(np.float64) - b[fin]) <= 1e-5 * np.linalg.norm(b[fin].astype(np.float64))
