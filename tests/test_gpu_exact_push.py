"""Exact searches whose levels push: up to 128 sources on symmetric graphs of a million arcs or
more, where a frontier of few arcs follows its own lists instead of scanning the graph.  Long
paths beside and into a dense component (a frontier that grows at a stroke), hubs on the way
(lists cut into tasks), nodes in any order, self-loops and repeated arcs.  Sums are the oracle's,
bit for bit; a component without a source costs a level next to nothing."""
import time

import numpy as np
import pytest

from test_gpu_exact import _check_sources, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _symmetric(hb, n, u, v, name):  # noqa: F811
    loop = u == v
    s, d = np.concatenate([u, v[~loop]]), np.concatenate([v, u[~loop]])
    order = np.lexsort((d, s))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(s, minlength=n), out=off[1:])
    return hb.Graph(off, d[order].astype(np.uint32), name)


def _graph(hb, kind):  # noqa: F811
    """The first nodes are a path, then come a random component and the stars' leaves."""
    rng = np.random.default_rng(23)
    path, core = 300, {"large": 140_000}.get(kind, 60_000)
    u, v = np.arange(path - 1), np.arange(1, path)
    cu, cv = path + rng.integers(0, core, 560_000), path + rng.integers(0, core, 560_000)
    hub = path + np.zeros(3000, np.int64)  # a node of more than one task
    cu, cv = np.concatenate([cu, hub]), np.concatenate([cv, path + rng.integers(0, core, 3000)])
    n = path + core
    u, v = np.concatenate([u, cu]), np.concatenate([v, cv])
    if kind in ("into", "shuffled"):  # the path ends in the component, at its hub
        u, v = np.append(u, path - 1), np.append(v, path)
    if kind in ("stars", "shuffled"):  # hubs along the path, each with 300 leaves of its own
        at = np.repeat(np.arange(20, path, 40), 300)
        u, v = np.concatenate([u, at]), np.concatenate([v, n + np.arange(at.size)])
        n += at.size
    if kind == "loops":
        u, v = np.concatenate([u, np.arange(0, path, 3), [5, 5, 6]]), np.concatenate([v, np.arange(0, path, 3), [6, 6, 5]])
    if kind == "shuffled":
        to = rng.permutation(n)
        u, v = to[u], to[v]
    return _symmetric(hb, n, u, v, kind)


@pytest.mark.parametrize("kind", ["beside", "into", "stars", "loops", "shuffled", "large"])
@pytest.mark.parametrize("lo,hi", [(0, 1), (3, 67), (150, 278), (299, 301), (290, 419)])
def test_pushed_levels_match_oracle(hb, oracle, kind, lo, hi):  # noqa: F811
    g = _graph(hb, kind)
    assert g.width() >= 1 << 20
    say("push", kind, lo, hi, g.size(), g.width())
    _check_sources(hb, oracle, g, lo, hi, (kind, lo, hi))


def test_a_component_without_a_source_is_not_scanned(hb):  # noqa: F811
    """A path of 1,500 nodes beside R-MAT-20 (some 30 M arcs): a level costs about what it does
    on the path alone; scanning the component in every level takes twenty times as long."""
    from sparkx_amd.exact import exact_bfs
    path, core = 1500, hb.Graph.rmat(20, 16, seed=2)
    line = _symmetric(hb, path, np.arange(path - 1), np.arange(1, path), "path")
    both = hb.Graph(np.concatenate([line.offsets, core.offsets[1:] + line.offsets[-1]]),
                    np.concatenate([line.neighbours, core.neighbours + np.uint32(path)]), "path and R-MAT-20")

    def searched(g, sources):
        t = time.perf_counter()
        r = exact_bfs(g, sources, inv_sum=False)
        return time.perf_counter() - t, r

    times = {}
    for g in (line, both):
        base = min(searched(g, (0, 0))[0] for _ in range(3))  # staging alone
        runs = [searched(g, (0, 64)) for _ in range(3)]
        assert all(np.array_equal(r[0], np.full(64, path)) for _, r in runs)
        times[g.name] = min(t for t, _ in runs) - base
    say("path alone", times["path"], "beside R-MAT-20", times[both.name])
    assert times[both.name] < 6 * times["path"]
