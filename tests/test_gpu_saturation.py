"""Saturated sketches (equal to the bound of all sketches) are not recomputed and end a
node's search for neighbours early; every result stays the oracle's, bit for bit.  The
graphs put the rule's exceptions together with a component that saturates: pairs of nodes
that only have each other, self-loops, repeated arcs, small components that keep the bound
out of reach, sinks of a directed graph, and hubs cut into chunks."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _csr(hb, n, src, dst, name):  # noqa: F811
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(src, minlength=n), out=off[1:])
    return hb.Graph(off, dst[order].astype(np.uint32), name)


def _graph(hb, kind):  # noqa: F811
    rng = np.random.default_rng(7)
    core = 1500
    s, d = rng.integers(0, core, 9000), rng.integers(0, core, 9000)
    if kind == "directed":  # heads without arcs of their own among them
        return _csr(hb, core + 200, s, rng.integers(0, core + 200, s.size), kind)
    n = core + 80
    extra = []
    if kind == "pairs":  # 20 pairs, 10 nodes with a self-loop, 30 isolated nodes
        extra = [(core + 2 * i, core + 2 * i + 1) for i in range(20)] + [(core + 40 + i,) * 2 for i in range(10)]
    elif kind == "triangles":  # in the bound, out of the component's reach
        for i in range(20):
            a = core + 3 * i
            extra += [(a, a + 1), (a + 1, a + 2), (a, a + 2)]
    elif kind == "doubled":  # pairs joined twice: two neighbours each, so part of the bound
        extra = [(core + 2 * i, core + 2 * i + 1) for i in range(10)] * 2
    elif kind == "hubs":
        extra = [(h, v) for h in (3, 700) for v in rng.choice(core, 900, replace=False) if v != h]
    e = np.array(extra, dtype=np.int64).reshape(-1, 2)
    u, v = np.concatenate([s, e[:, 0]]), np.concatenate([d, e[:, 1]])
    loop = u == v
    return _csr(hb, n, np.concatenate([u, v[~loop]]), np.concatenate([v, u[~loop]]), kind)


@pytest.mark.parametrize("kind", ["pairs", "triangles", "doubled", "hubs", "directed"])
@pytest.mark.parametrize("p", [4, 6, 7, 8, 10, 11, 13])
def test_saturation_matches_oracle(hb, oracle, kind, p):  # noqa: F811
    g = _graph(hb, kind)
    say("saturation", kind, p, g.size(), g.width())
    ref = _oracle_run(oracle, g, p)
    for kw in (dict(layout="degree"), dict(layout="input"), dict(layout="degree", schedule=(2, 16, 64)),
               dict(layout="degree", graph_capture=True), dict(layout="degree", max_iters=3)):
        want = _oracle_run(oracle, g, p, max_iters=3) if "max_iters" in kw else ref
        with hb.HyperBall(g, p, **kw) as h:
            _assert_same(h, want, oracle, p, f"{kind} p={p} {kw}")
            scanned = sum(h.stats.kernel_arcs[s] for s in range(4))
        if p <= 10 and kind in ("pairs", "hubs") and kw == dict(layout="degree"):
            # the search ends early for most nodes of the iterations after saturation
            with hb.HyperBall(g, p, dense=True, **kw) as full:
                assert scanned < 0.9 * sum(full.stats.kernel_arcs[s] for s in range(4))


def test_saturation_of_trivial_graphs(hb, oracle):  # noqa: F811
    """One node with self-loops, one pair, a complete graph: the bound is reached at once."""
    one = _csr(hb, 1, np.zeros(3, np.int64), np.zeros(3, np.int64), "one")
    pair = _csr(hb, 2, np.array([0, 1]), np.array([1, 0]), "pair")
    k = np.arange(40)
    s, d = [a.ravel() for a in np.meshgrid(k, k)]
    full = _csr(hb, 40, s[s != d], d[s != d], "complete")
    for g in (one, pair, full):
        for p in (4, 7):
            say("trivial", g.name, p)
            ref = _oracle_run(oracle, g, p)
            with hb.HyperBall(g, p, layout="degree") as h:
                _assert_same(h, ref, oracle, p, f"{g.name} p={p}")


def test_saturation_in_a_batch(hb, oracle):  # noqa: F811
    """Every graph of a batch has its own bound and its own symmetric flag."""
    from sparkx_amd import _lib
    from sparkx_amd.batch import HyperBallBatch
    kinds = ["pairs", "triangles", "doubled", "hubs", "directed"]
    items = [(_graph(hb, kind), p) for p in (4, 5, 6, 7, 8) for kind in kinds]
    items += [(hb.Graph.rmat(12, 16, seed=4), 7), (hb.Graph.rmat(12, 16, seed=5), 8)]  # hub chunks
    b = HyperBallBatch(items)
    try:
        for kw in (dict(), dict(graph_capture=False), dict(dense=True), dict()):
            b.run(**kw)
            for i, (g, p) in enumerate(items):
                say("batch", kw, i, g.name, p)
                ref = _oracle_run(oracle, g, p)
                it, _, inc = b.graph_stats(i)
                assert it == ref.iterations and list(inc) == list(ref.increases)
                dist, inv = b.accumulators(i)
                assert np.array_equal(dist, ref.dist) and np.array_equal(inv, ref.inv)
                assert np.array_equal(b.registers(i, _lib.HB_REGS_REFERENCE).ravel(), ref.regs_ref)
                assert np.array_equal(b.registers(i, _lib.HB_REGS_LATEST).ravel(), ref.regs_last)
    finally:
        b.close()
