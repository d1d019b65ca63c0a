"""Walk-count inputs at the lengths where a pass changes its way through a list: the 64 arcs of
a lane, the 512 arcs of a tile of 64 short lists, the 256 arcs of a wavefront's turn and the
2,048 of a hub's chunk; short lists alone, of one length, and among long ones, the last
wavefront partly filled.  The counts are exact, so each logarithm is within 1 f32 ulp of the
oracle's (the two log1p may differ in the last f64 bit) and a difference of two within 1e-6
relative + 1e-9."""
import numpy as np
import pytest

from test_gpu_walks import _csr, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu

LISTS = {
    "one length, a tile": [8] * 64,
    "one length, a tile and one arc": [8] * 63 + [9],
    "longest short lists": [64] * 130,
    "short, odd": [0, 1, 63, 64, 5, 0, 0, 31, 33] * 15,
    "the lines": [64, 65, 255, 256, 257, 0, 1] * 10,
    "chunks": [2047, 2048, 2049, 4096, 4097, 3, 60, 100],
    "one node": [1],
}


@pytest.mark.parametrize("layout", ["input", "degree"])
@pytest.mark.parametrize("kind", list(LISTS))
def test_walk_lists(hb, oracle, kind, layout):  # noqa: F811
    from sparkx_amd.surrogate import walk_features
    deg = np.array(LISTS[kind])
    n = deg.size
    rng = np.random.default_rng(n)
    off, nb = _csr(n, np.repeat(np.arange(n), deg), rng.integers(0, n, deg.sum()))
    g = hb.Graph(off, nb, "lists")
    for passes, diff in ((2, [4, 5]), (3, [5])):
        say("walk lists", kind, layout, passes)
        want = oracle.walk_inputs(g.offsets, g.neighbours, passes)
        logs = [k for k in range(6) if k not in diff]
        with hb.HyperBall(g, 4, _run=False, layout=layout) as h:
            got, _ = walk_features(h, passes)
        np.testing.assert_array_max_ulp(got[:, logs], want[:, logs], maxulp=1)
        np.testing.assert_allclose(got[:, diff], want[:, diff], rtol=1e-6, atol=1e-9)
