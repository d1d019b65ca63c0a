"""A node whose sketch is the bound after iteration 1, with no neighbour that changed then, is
not counted as changed when a neighbour saturates later: the next iteration is scheduled from
the nodes that did change."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _graph(hb, oracle, p, n=4096):  # noqa: F811
    """Directed.  "top" nodes hold every register's maximum and "rest" nodes fill up; both have
    a self-loop only.  x and the "full" nodes list all top nodes: they are the bound after
    iteration 1.  v, whose register is x's, lists x: unchanged by iteration 1, saturated in 2.
    "late" nodes, with v's register, list v: they change in iteration 3, and no node lists one."""
    idx, rank = np.array([oracle.index_rank(p, i) for i in range(n)]).T
    order = np.lexsort((np.arange(n), -rank, idx))
    top = order[np.r_[True, np.diff(idx[order]) != 0]]
    free = np.setdiff1d(np.arange(n), top)
    reg = np.bincount(idx[free][rank[free] == 1]).argmax()
    v, x = free[(idx[free] == reg) & (rank[free] == 1)][:2]
    same = np.setdiff1d(free[idx[free] == reg], [v, x])
    late = same[:max(1, min(same.size, n // 20))]
    other = np.setdiff1d(free, np.r_[v, x, late])
    full = other[:int(0.5 * n) - late.size // 2]
    lists = {int(u): [int(u)] for u in np.r_[top, other[full.size:]]}
    for u in full:
        lists[int(u)] = [int(v), *top.tolist()]
    lists[int(x)] = top.tolist()
    lists[int(v)] = [int(x)] * (n // 4)
    for u in late:
        lists[int(u)] = [int(v)]
    off = np.zeros(n + 1, np.uint64)
    np.cumsum([len(lists[u]) for u in range(n)], out=off[1:])
    g = hb.Graph(off, np.concatenate([lists[u] for u in range(n)]).astype(np.uint32), "bound")
    assert 2 * (full.size + 1) <= n < 2 * (full.size + late.size)  # not enough changed; enough if miscounted
    return g


@pytest.mark.parametrize("p", [4, 5, 6])
def test_bound_reached_in_the_first_iteration(hb, oracle, p):  # noqa: F811
    g = _graph(hb, oracle, p)
    say("bound at once", p, g.size(), g.width())
    ref = _oracle_run(oracle, g, p)
    assert ref.iterations == 4
    for kw in (dict(layout="input"), dict(layout="input", graph_capture=True)):
        with hb.HyperBall(g, p, **kw) as h:
            _assert_same(h, ref, oracle, p, f"p={p} {kw}")
            assert h.stats.iter_nodes[3] == 0, kw  # no node lists one that changed in iteration 3
