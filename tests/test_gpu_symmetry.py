"""The symmetry of a staged graph, found from fingerprints of its arcs and of their reverses,
at the edges of the 512 arcs that a wavefront takes at a time: the answer is that of the
sorted arc lists, with empty nodes between, before and after the others, hubs whose arcs span
several wavefronts, repeated arcs and self-loops."""
import numpy as np
import pytest

from test_gpu_parity import hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _arcs(kind, pairs):
    rng = np.random.default_rng(pairs)
    if kind == "path":
        u, v = np.arange(pairs), np.arange(pairs) + 1
    elif kind == "hub":
        u, v = np.full(pairs, 5), np.arange(pairs) + 6
    elif kind == "empty runs":  # 300 empty nodes before, between each two and after the others
        u, v = 300 * (1 + rng.integers(0, 40, pairs)), 300 * (41 + rng.integers(0, 40, pairs))
    else:  # few nodes: repeated arcs; loops
        u, v = rng.integers(0, 9, pairs), rng.integers(0, 9, pairs)
    return np.concatenate([u, v[u != v]]), np.concatenate([v, u[u != v]])


@pytest.mark.parametrize("kind", ["path", "hub", "empty runs", "repeated"])
@pytest.mark.parametrize("pairs", [1, 31, 255, 256, 257, 511, 2048, 40000])
def test_symmetry(hb, kind, pairs):  # noqa: F811
    u, v = _arcs(kind, pairs)
    n = int(max(u.max(), v.max())) + 301
    moved = v.copy()
    moved[-1] = (moved[-1] + 1) % n  # one arc ends a node further on
    for s, d in ((u, v), (u, moved)):
        order = np.lexsort((d, s))
        off = np.zeros(n + 1, np.uint64)
        np.cumsum(np.bincount(s, minlength=n), out=off[1:])
        back = np.lexsort((s, d))
        want = bool((s[order] == d[back]).all() and (d[order] == s[back]).all())
        say("symmetry", kind, pairs, want)
        g = hb.Graph(off, d[order].astype(np.uint32), kind)
        with hb.HyperBall(g, 4, max_iters=1) as h:
            assert bool(h.stats.symmetric) == want
