"""Exact searches of directed graphs.  Up to 128 sources follow the arcs as they are; more search
the reversed arcs, unless those find no memory.  Sums are the oracle's, bit for bit, whichever
way; a search that reaches little does not pay for reversing the graph."""
import ctypes as C
import time

import numpy as np
import pytest

from test_gpu_exact import _check_sources, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _directed(hb, n, s, d, name):  # noqa: F811
    order = np.lexsort((d, s))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(s, minlength=n), out=off[1:])
    return hb.Graph(off, d[order].astype(np.uint32), name)


def _graph(hb, kind):  # noqa: F811
    rng = np.random.default_rng(31)
    n = 4357
    if kind == "random":
        return _directed(hb, n, rng.integers(0, n, 9000), rng.integers(0, n, 9000), kind)
    if kind == "hubs":  # lists out and in of several tasks, loops, repeated arcs
        s = np.concatenate([np.zeros(n, np.int64), np.full(1500, 9), rng.integers(0, n, 6000), np.arange(3000), [7, 7]])
        d = np.concatenate([np.arange(n), rng.integers(0, n, 1500), rng.integers(0, n, 6000), np.full(3000, 40), [8, 8]])
        return _directed(hb, n, s, d, kind)
    # a path of 200 nodes into a component, no arc back: more levels than are kept
    s = np.concatenate([np.arange(200), rng.integers(200, n, 20000)])
    d = np.concatenate([np.arange(1, 201), rng.integers(200, n, 20000)])
    return _directed(hb, n, s, d, kind)


@pytest.mark.parametrize("kind", ["random", "hubs", "into"])
@pytest.mark.parametrize("lo,hi", [(0, 1), (5, 69), (130, 258), (0, 129), (3, 700)])
@pytest.mark.parametrize("limit", [None, 2_000_000])
def test_directed_matches_oracle(hb, oracle, monkeypatch, kind, lo, hi, limit):  # noqa: F811
    g = _graph(hb, kind)
    if limit:  # less than the reversed arcs and the sort's memory take, enough for one slice
        g = _directed(hb, g.size(), np.concatenate([np.repeat(np.arange(g.size()), g.degrees()),
                                                    np.full(200_000, g.size() - 2)]),
                      np.concatenate([g.neighbours.astype(np.int64), np.full(200_000, g.size() - 1)]), kind)
        monkeypatch.setenv("SPARKX_HB_BFS_BYTES", str(limit))
    say("directed", kind, lo, hi, limit, g.size(), g.width())
    _check_sources(hb, oracle, g, lo, hi, (kind, lo, hi, limit))


def test_large_directed_graph_is_not_reversed_for_one_source(hb):  # noqa: F811
    """From the head of a path of four nodes beside 16 M arcs: about as long as on a path there and
    back, whose arcs need no reversing (that takes some ten times as long as the search)."""
    from sparkx_amd import _lib
    L = _lib.load()
    rng = np.random.default_rng(2)
    n, m = 1 << 20, 16 << 20
    s, d = rng.integers(4, n, m), rng.integers(4, n, m)
    path = np.arange(3)

    def best(s, d):
        g = _directed(hb, n, np.concatenate([path, s]), np.concatenate([path + 1, d]), "path")
        off, nb = g.offsets, g.neighbours
        ctx, reach, times = C.c_void_p(), np.zeros(1, np.uint64), []
        _lib.check(L.hb_create(C.byref(ctx), 0))
        try:
            _lib.check(L.hb_set_layout(ctx, _lib.HB_LAYOUT_INPUT))
            _lib.check(L.hb_stage_csr(ctx, off.ctypes.data, off.itemsize, n, nb.ctypes.data, nb.itemsize, g.width()))
            for _ in range(5):
                t = time.perf_counter()
                _lib.check(L.hb_exact_bfs(ctx, 0, 1, _lib.ptr(reach, C.c_uint64), None, None))
                times.append(time.perf_counter() - t)
        finally:
            L.hb_destroy(ctx)
        return min(times), int(reach[0])

    one, reached = best(s, d)
    assert reached == 3
    alone, _ = best(path + 1, path)
    say("beside 16 M arcs", one, "alone", alone)
    assert one < 3 * alone


def test_long_runs_of_nodes_without_arcs_to_them(hb, oracle):  # noqa: F811
    """129 sources of a directed graph of a million nodes, few of which are heads: the offsets of
    the reversed arcs do not wait for one thread to cross the gaps."""
    from sparkx_amd.exact import exact_bfs
    n = 1 << 20
    s = np.arange(300)
    g = _directed(hb, n, s, np.where(s < 150, 0, n - 300 + s), "gaps")
    say("gaps", g.size(), g.width())
    _check_sources(hb, oracle, g, 0, 129, "gaps")
    spread = _directed(hb, n, s, s * 3400 + 7, "spread")
    times = {}
    for x in (spread, g):
        runs = []
        for _ in range(4):
            t = time.perf_counter()
            exact_bfs(x, (0, 129), inv_sum=False)
            runs.append(time.perf_counter() - t)
        times[x.name] = min(runs)
    say(times)
    assert times["gaps"] < 3 * times["spread"]
