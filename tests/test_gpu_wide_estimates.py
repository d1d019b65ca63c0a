"""Estimates of register rows at p = 11..16 whose f32 sum of 2^-M rounds: the reference adds
register after register, and the estimate is the oracle's bit for bit wherever the small terms
stand (early, late, in one lane's 16 registers or spread), across binades, with registers beyond
24 and beyond 35, with no zero register and with few.  And runs whose estimates pass linear
counting, so that a row of more than one pass is read back."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_parity import _assert_same, _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def _rows(p):
    m, top = 1 << p, 64 - p + 1
    rng = np.random.default_rng(p)
    rows = []

    def ranks(load):  # registers after about load * m insertions
        u = rng.random(m) ** (1.0 / max(load, 1e-3))  # P(rank <= k) = (1 - 2^-k)^load
        return np.clip(np.ceil(-np.log2(1.0 - u + 1e-300)), 0, top).astype(np.uint8)

    for load in (3, 6, 20, 100, 1e4, 1e6, 1e9, 1e12):
        rows += [ranks(load) for _ in range(3)]
    for v in (1, 2, 5, 11, 20, 23, 24, 25, 30, 34, 35, 36, top):
        rows.append(np.full(m, v, np.uint8))
    for base in (1, 2, 4, 9, 14):
        for tiny in (20, 23, 24, 26, 29, 33, 35, 36, top):
            for where in (slice(0, 5), slice(0, 1030), slice(m - 7, m), slice(m // 2 - 3, m // 2 + 3), slice(5, None, 16),
                          slice(1, None, 97), slice(3, None, 1024)):
                r = np.full(m, base, np.uint8)
                r[where] = min(tiny, top)
                rows.append(r)
    for _ in range(40):  # any values, few zeros among them
        lo, hi = sorted(rng.integers(1, top + 1, 2))
        r = rng.integers(lo, hi + 1, m).astype(np.uint8)
        if rng.random() < 0.5:
            r[rng.integers(0, m, rng.integers(1, 30))] = 0
        rows.append(r)
    for _ in range(20):  # descending and ascending runs: the sum grows through many binades
        r = np.sort(ranks(10.0 ** rng.uniform(0.5, 9)))
        rows += [r, r[::-1]]
    return np.stack(rows)


@pytest.mark.parametrize("p", [11, 12, 13, 14, 15, 16])
def test_estimates_of_crafted_rows(hb, oracle, p):  # noqa: F811
    from sparkx_amd import _lib
    rows = np.ascontiguousarray(_rows(p))
    n = len(rows)
    say("crafted rows", p, n)
    off = np.arange(n + 1, dtype=np.uint64)  # a self-loop each
    g = hb.Graph(off, np.arange(n, dtype=np.uint32), "rows")
    zeros = np.zeros(n)
    with hb.HyperBall(g, p, layout="input", _run=False) as h:
        _lib.check(h._L.hb_restore(h._ctx, p, _lib.ptr(rows, C.c_uint8), _lib.ptr(zeros, C.c_double),
                                   _lib.ptr(zeros, C.c_double)))
        h._ran(None)
        got = h.estimates(_lib.HB_REGS_REFERENCE)
    want = oracle.estimates(p, rows)
    bad = np.nonzero(got.view(np.uint32) != want.view(np.uint32))[0]
    assert bad.size == 0, (p, bad[:10], got[bad[:10]], want[bad[:10]])


@pytest.mark.parametrize("p,n", [(13, 9001), (14, 13001), (15, 23001)])
def test_runs_beyond_linear_counting(hb, oracle, p, n):  # noqa: F811
    """A component of more nodes than linear counting is used up to."""
    g = hb.Graph.erdos_renyi(n, 3 * n, seed=p)
    say("beyond linear counting", p, n, g.width())
    ref = _oracle_run(oracle, g, p)
    assert oracle.estimates(p, ref.regs_ref).max() > {13: 6500, 14: 11500, 15: 20000}[p]
    with hb.HyperBall(g, p) as h:
        _assert_same(h, ref, oracle, p, f"p={p}")
