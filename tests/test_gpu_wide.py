"""Precisions 11..16 (one wavefront per node and 1 KiB chunk of the row): list lengths at
the edges of a wavefront's ids, of the hash pass and of the hub tasks; sums that are exact,
that round, and that round below the final binade.  Registers, estimates and accumulators
are the oracle's, bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 3, 4, 63, 64, 65, 128, 255, 256, 257, 511, 512, 513, 1025]


def _graph(hb, n, seed, directed=False):  # noqa: F811
    """Node k of the first ones has exactly EDGES[k] arcs out; the rest is sparse."""
    rng = np.random.default_rng(seed)
    src = np.repeat(np.arange(len(EDGES)), EDGES)
    dst = np.concatenate([rng.choice(np.arange(20, n), d, replace=False) for d in EDGES])
    a, b = rng.integers(20, n, 3 * n), rng.integers(20, n, 3 * n)
    src, dst = np.concatenate([src, a]), np.concatenate([dst, b])
    if not directed:
        src, dst = np.concatenate([src, dst[src != dst]]), np.concatenate([dst, src[src != dst]])
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(src, minlength=n), out=off[1:])
    return hb.Graph(off, dst[order].astype(np.uint32), f"edges{n}")


@pytest.mark.parametrize("p", [11, 12, 13, 14, 16])
@pytest.mark.parametrize("directed", [False, True])
def test_wide_rows_at_list_edges(hb, oracle, p, directed):  # noqa: F811
    g = _graph(hb, 1500 if p < 14 else 1100, p, directed)
    say("wide edges", p, directed, g.size(), g.width())
    ref = _oracle_run(oracle, g, p)
    for kw in (dict(), dict(dense=True), dict(layout="input"), dict(graph_capture=True), dict(layout="chain")):
        with hb.HyperBall(g, p, **kw) as h:
            _assert_same(h, ref, oracle, p, f"p={p} {kw}")
            assert h.stats.kernel_items[3] == sum(-(-d // 256) for d in EDGES if d > 256)  # tasks


@pytest.mark.parametrize("p", [11, 12])
def test_wide_sums_beyond_exact(hb, oracle, p):  # noqa: F811
    """Sketches of 200,000 nodes: sums with registers far below the final binade's ulp, in
    every iteration up to the last (the oracle sums them one by one)."""
    g = hb.Graph.erdos_renyi(200_001, 500_000, seed=p)
    say("wide sums", p, g.size(), g.width())
    ref = _oracle_run(oracle, g, p)
    with hb.HyperBall(g, p) as h:
        _assert_same(h, ref, oracle, p, f"p={p}")
