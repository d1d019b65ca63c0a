"""Exact searches in slices of up to 2,048 sources: rows of every width, source ranges
that end inside a word, a row or a slice, lists cut into hub tasks, reversed arcs of
directed graphs, and harmonic sums whose binades change at every chunk boundary or that
need more levels than are kept.  Integer sums and harmonic sums are the oracle's, bit for
bit."""
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
    rng = np.random.default_rng(11)
    n = 4357  # not a multiple of a chunk
    if kind == "dense":
        s, d = rng.integers(0, n, 40000), rng.integers(0, n, 40000)
    elif kind == "sparse":  # about 12 levels, unreached nodes
        s, d = rng.integers(0, n, 4500), rng.integers(0, n, 4500)
    elif kind == "hubs":  # in-lists of more than one task
        s = np.concatenate([np.zeros(n - 1, np.int64), np.full(1500, 9), rng.integers(0, n, 6000)])
        d = np.concatenate([np.arange(1, n), rng.integers(10, n, 1500), rng.integers(0, n, 6000)])
    else:  # "long": more levels than are kept
        s = np.arange(n - 1)
        d = s + 1
        far = rng.integers(0, n - 60, 300)
        s, d = np.concatenate([s, far]), np.concatenate([d, far + rng.integers(1, 60, 300)])
    if kind == "hubs":
        return _csr(hb, n, s, d, kind + " directed")
    return _csr(hb, n, np.concatenate([s, d[s != d]]), np.concatenate([d, s[s != d]]), kind)


@pytest.mark.parametrize("kind", ["dense", "sparse", "hubs", "long"])
@pytest.mark.parametrize("lo,hi", [(0, 1), (3, 67), (100, 229), (7, 600), (1, 1026), (0, 2049), (128, 4357)])
def test_slices_match_oracle(hb, oracle, kind, lo, hi):  # noqa: F811
    if kind == "long" and hi - lo > 700:
        pytest.skip("the oracle's long searches take minutes")
    g = _graph(hb, kind)
    say("slices", kind, lo, hi, g.size(), g.width())
    _check_sources(hb, oracle, g, lo, hi, (kind, lo, hi))


def test_symmetric_hubs_in_a_slice(hb, oracle):  # noqa: F811
    g = hb.Graph.rmat(13, 16, seed=3)
    say("rmat13 slice", g.size(), g.width(), int(g.degrees().max()))
    assert g.degrees().max() > 1024
    _check_sources(hb, oracle, g, 11, 2400, "rmat13")
