"""kernel_first_nodes counts the nodes whose own register block iteration 1 does not read:
those of the bins that hash ids with p <= 10.  Wide rows (p > 10) hash the neighbours' ids only."""
import pytest

from test_gpu_parity import hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [4, 6, 10, 11, 12, 16])
def test_first_iteration_nodes_and_arcs(hb, p):  # noqa: F811
    g = hb.Graph.erdos_renyi(700, 4200, seed=2)
    say("first iteration", p, g.size(), g.width())
    with hb.HyperBall(g, p, layout="degree") as h:
        st = h.stats
        linked = int((g.degrees() > 0).sum())
        assert sum(st.kernel_first_arcs[:3]) == g.width()  # no list is long enough to be cut
        assert sum(st.kernel_first_nodes[:3]) == (linked if p <= 10 else 0)
        assert st.iter_nodes[0] == linked
