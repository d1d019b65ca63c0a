"""Copies between host arrays and the device: sizes around the line between one copy and the
pinned slots (4 MiB), 4- and 8-byte ids and offsets, refused ids at either end, and several threads
staging and reading at once, of which one at a time holds the slots."""
import ctypes as C
import threading

import numpy as np
import pytest

from test_gpu_parity import hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _ring(n, extra, seed, off_type=np.uint64, id_type=np.uint32):
    """Every node lists the next one, the first `extra` nodes a random one too."""
    rng = np.random.default_rng(seed)
    deg = np.ones(n, np.int64)
    deg[:extra] = 2
    off = np.zeros(n + 1, off_type)
    np.cumsum(deg, out=off[1:])
    nbr = np.empty(n + extra, id_type)
    nbr[off[:-1].astype(np.int64)] = (np.arange(n) + 1) % n
    nbr[off[:extra].astype(np.int64) + 1] = rng.integers(0, n, extra)
    return off, nbr


def _staged(off, nbr):
    from sparkx_amd import _lib
    L, ctx = _lib.load(), C.c_void_p()
    _lib.check(L.hb_create(C.byref(ctx), 0))
    try:
        _lib.check(L.hb_set_layout(ctx, _lib.HB_LAYOUT_INPUT))
        rc = L.hb_stage_csr(ctx, off.ctypes.data, off.itemsize, off.size - 1, nbr.ctypes.data, nbr.itemsize, nbr.size)
        message = L.hb_last_error().decode()
        o, v = np.full(off.size, -1, np.int64).view(np.uint64), np.full(nbr.size, -1, np.int64).view(np.uint64)
        if rc == 0:
            _lib.check(L.hb_read_csr(ctx, _lib.ptr(o, C.c_uint64), _lib.ptr(v, C.c_uint64)))
        return rc, message, o, v
    finally:
        L.hb_destroy(ctx)


@pytest.mark.parametrize("arcs", [1, 1000, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, (1 << 22) + 12_345, 9_000_001])
@pytest.mark.parametrize("wide", [False, True])
def test_csr_round_trip(hb, arcs, wide):  # noqa: F811
    n = max(1, arcs // 2 + 1)
    off, nbr = _ring(n, arcs - n, arcs, np.uint64 if wide else np.uint32, np.uint64 if wide else np.uint32)
    say("csr", arcs, wide)
    rc, message, o, v = _staged(off, nbr)
    assert rc == 0, message
    assert np.array_equal(o, off.astype(np.uint64)) and np.array_equal(v, nbr.astype(np.uint64))
    for at in (0, arcs // 2, arcs - 1):
        bad = nbr.copy()
        bad[at] = n
        rc, message, _, _ = _staged(off, bad)
        assert rc == -1 and f"neighbour {n} at arc {at} " in message  # HB_EINVAL, the first such arc


@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 20) + 1])
@pytest.mark.parametrize("layout", ["input", "degree"])
def test_results_of_either_size_agree(hb, n, layout):  # noqa: F811
    """Arrays of 4 and 8 bytes a node on either side of the line: equal to the same nodes' values
    of a run whose arrays all go in one copy."""
    off, nbr = _ring(n, 0, 1)  # symmetric under rotation but for the hashes
    g = hb.Graph(off, nbr, "ring")
    say("results", n, layout)
    with hb.HyperBall(g, 4, layout=layout, max_iters=3) as h:
        dist, est, regs = h.geodesic_distances(), h.estimates(), h.registers()
        closeness = h.compute_closeness_centrality(False)
    part = 20_000  # after three iterations a node depends on the three after it only
    short = hb.Graph(np.arange(part + 4, dtype=np.uint64),
                     np.minimum(np.arange(1, part + 4), part + 2).astype(np.uint32), "part")
    with hb.HyperBall(short, 4, layout=layout, max_iters=3) as h:
        assert np.array_equal(h.geodesic_distances()[:part], dist[:part])
        assert np.array_equal(h.estimates()[:part], est[:part])
        assert np.array_equal(h.registers()[:part], regs[:part])
    assert closeness.shape == (n,) and np.isfinite(closeness).all()


def test_threads_share_the_slots(hb):  # noqa: F811
    """Six threads stage graphs of some 12 MB, read them back and read results, all at once."""
    graphs = [_ring(600_000 + 7 * i, 500_000, i) for i in range(6)]
    want = []
    for off, nbr in graphs:
        with hb.HyperBall(hb.Graph(off, nbr, "ring"), 4, max_iters=4) as h:
            want.append((h.geodesic_distances(), h.estimates()))
    failures = []

    def work(i):
        try:
            off, nbr = graphs[i]
            for _ in range(3):
                rc, message, o, v = _staged(off, nbr)
                assert rc == 0, message
                assert np.array_equal(o, off) and np.array_equal(v, nbr)
                with hb.HyperBall(hb.Graph(off, nbr, "ring"), 4, max_iters=4) as h:
                    assert np.array_equal(h.geodesic_distances(), want[i][0])
                    assert np.array_equal(h.estimates(), want[i][1])
        except BaseException as e:  # noqa: BLE001 - reported by the test's own thread
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(graphs))]
    say("threads", len(threads))
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
