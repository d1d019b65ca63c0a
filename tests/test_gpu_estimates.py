"""Estimates read after a run: those the run left where they belong to the buffer that is
asked for, else computed from its rows; for both buffers, runs that converge and runs cut off
at odd and even iterations, they are the oracle's estimates of the rows that are read."""
import numpy as np
import pytest

from test_gpu_parity import _oracle_run, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [4, 6, 8, 10, 11, 13])
@pytest.mark.parametrize("layout", ["degree", "input"])
def test_estimates_of_both_buffers(hb, oracle, p, layout):  # noqa: F811
    from sparkx_amd import _lib
    g = hb.Graph.erdos_renyi(2000, 3500, seed=p)  # isolated nodes, small components
    for it in (1, 2, 3, 6, 0):
        say("estimates", p, layout, it)
        ref = _oracle_run(oracle, g, p, max_iters=it)
        with hb.HyperBall(g, p, layout=layout, max_iters=it) as h:
            for which, regs in ((_lib.HB_REGS_REFERENCE, ref.regs_ref), (_lib.HB_REGS_LATEST, ref.regs_last)):
                assert np.array_equal(h.estimates(which), oracle.estimates(p, regs))


def test_estimates_of_a_batch(hb, oracle):  # noqa: F811
    from sparkx_amd import _lib
    from sparkx_amd.batch import HyperBallBatch
    graphs = [(hb.Graph.erdos_renyi(1500, 2500, seed=p), p) for p in (4, 5, 6, 7, 8)]
    for it in (1, 2, 3, 0):
        with HyperBallBatch(graphs, max_iters=it) as bt:
            bt.run()
            for i, (g, p) in enumerate(graphs):
                ref = _oracle_run(oracle, g, p, max_iters=it)
                for which, regs in ((_lib.HB_REGS_REFERENCE, ref.regs_ref), (_lib.HB_REGS_LATEST, ref.regs_last)):
                    assert np.array_equal(bt.estimates(i, which), oracle.estimates(p, regs)), (it, p, which)
