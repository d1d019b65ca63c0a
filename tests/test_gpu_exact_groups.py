"""Exact searches in several groups of slices: little memory per group, so that groups follow
each other in the same buffers, the last one shorter than they are; searches that turn out longer
than the levels kept after earlier groups have delivered; slices and rows halved until they fit.
Also the u16 distances of long searches at every row width and in more than one slice.  Sums are
the oracle's, bit for bit."""
import numpy as np
import pytest

from test_gpu_exact import _check_sources, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _csr(hb, n, src, dst, name):  # noqa: F811
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(np.bincount(src, minlength=n), out=off[1:])
    return hb.Graph(off, dst[order].astype(np.uint32), name)


def _graph(hb, kind):  # noqa: F811
    rng = np.random.default_rng(17)
    if kind == "ladder":  # 24 rungs of 60 nodes, arcs within a rung and to the next: some 30 levels
        w, rungs = 60, 24
        n = w * rungs
        a = rng.integers(0, n, 3 * n)
        b = a // w * w + rng.integers(0, w, a.size)
        up = np.arange(n - w)
        s, d = np.concatenate([a, up[::7]]), np.concatenate([b, up[::7] + w])
    elif kind == "then long":  # the first 1,500 nodes are close to each other, the rest is a path
        core, path = 1500, 300
        n = core + path
        s = np.concatenate([rng.integers(0, core, 9000), np.arange(core, n - 1)])
        d = np.concatenate([rng.integers(0, core, 9000), np.arange(core + 1, n)])
    else:  # lists in and out of several tasks
        n = 2900
        s = np.concatenate([np.zeros(1300, np.int64), rng.integers(0, n, 6000)])
        d = np.concatenate([np.arange(1, 1301), rng.integers(0, n, 6000)])
        if kind == "directed":
            return _csr(hb, n, s, d, kind)
    loop = s == d
    return _csr(hb, n, np.concatenate([s, d[~loop]]), np.concatenate([d, s[~loop]]), kind)


# bytes of a group: two words a row and one slice up to a row of 32 words in one slice
@pytest.mark.parametrize("kind", ["ladder", "then long", "hubs", "directed"])
@pytest.mark.parametrize("limit", [1_000_000, 2_000_000, 5_000_000, 14_000_000])
def test_groups_match_oracle(hb, oracle, monkeypatch, kind, limit):  # noqa: F811
    g = _graph(hb, kind)
    monkeypatch.setenv("SPARKX_HB_BFS_BYTES", str(limit))
    for lo, hi in ((0, g.size()), (1001, min(g.size(), 2300))):
        say("groups", kind, limit, lo, hi, g.size(), g.width())
        _check_sources(hb, oracle, g, lo, hi, (kind, limit, lo, hi))


@pytest.mark.parametrize("lo,hi", [(0, 1440), (3, 700), (9, 1200), (700, 830)])
def test_long_searches_of_many_sources(hb, oracle, lo, hi):  # noqa: F811
    g = _graph(hb, "ladder")
    say("ladder", lo, hi, g.size(), g.width())
    r, t, _ = _check_sources(hb, oracle, g, lo, hi, (lo, hi))
    assert (t[r > 0] / r[r > 0]).max() > 12  # more levels than are kept


def test_too_little_memory_is_reported(hb, monkeypatch):  # noqa: F811
    monkeypatch.setenv("SPARKX_HB_BFS_BYTES", "1000")
    from sparkx_amd.exact import ExactClosenessCentrality
    with pytest.raises(hb.HyperBallError) as e:
        ExactClosenessCentrality(_graph(hb, "hubs"), True)
    assert e.value.code == -2  # HB_ENOMEM


def test_distances_of_one_word_at_a_time(hb, oracle, monkeypatch):  # noqa: F811
    """Memory for the distances of 64 sources of a long search but not of 128: 64 at a time."""
    g = _graph(hb, "ladder")
    n = g.size()
    monkeypatch.setenv("SPARKX_HB_BFS_BYTES", str(n * 250))  # 51 bytes a node and 128 per 64 sources
    for lo, hi in ((0, 1), (5, 69), (100, 400)):
        say("one word", lo, hi, n)
        _check_sources(hb, oracle, g, lo, hi, (lo, hi))
