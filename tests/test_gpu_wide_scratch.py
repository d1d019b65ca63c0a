"""Hub tasks at p = 16 where 256-arc tasks would need more partial rows than are allowed
(dense graphs): tasks are longer, their rows stay within the bound, and the results are the
oracle's, bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def test_dense_graph_at_p16(hb, oracle):  # noqa: F811
    n, p = 2100, 16
    nbr = np.tile(np.arange(n, dtype=np.uint32), (n, 1))
    keep = ~np.eye(n, dtype=bool)
    keep[:, 1500:] &= (np.arange(n) % 8 > 0)[:, None]  # lists of 1,500 and of 2,099 arcs
    off = np.zeros(n + 1, np.uint64)
    np.cumsum(keep.sum(1), out=off[1:])
    g = hb.Graph(off, nbr[keep], "dense")
    say("dense p=16", g.size(), g.width())
    room = 1 << 30
    assert sum(-(-int(d) // 256) for d in g.degrees()) << p > room
    ref = _oracle_run(oracle, g, p)
    for kw in (dict(), dict(dense=True), dict(layout="input")):
        with hb.HyperBall(g, p, **kw) as h:
            assert 0 < h.stats.kernel_items[3] << p <= room, kw
            _assert_same(h, ref, oracle, p, f"{kw}")
