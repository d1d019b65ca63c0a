"""The network's gradient at sample counts around a wavefront's 16-sample tile, a block's four
tiles and the grid's 512 blocks, against the f64 oracle.  An f32 pre-activation may round to
the other bf16 neighbour than the oracle's, which moves that sample's share of a gradient by one
bf16 step (2^-8 of it): 5e-3 of the gradient's scale bounds it also where few samples share the
sum, and 2e-4 holds for 1,000 and more, as for the gradient's other test."""
import numpy as np
import pytest

from test_gpu_parity import _mlp_case, hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 63, 64, 65, 1000, 32767, 32769])
def test_gradient_at_tile_edges(hb, count):  # noqa: F811
    from oracle import mlp_oracle as M
    from sparkx_amd.surrogate import Surrogate
    params, norm, x, t = _mlp_case(seed=9, n=max(count, 1000))  # one sample has no deviation
    x, t = x[:count], t[:count]
    s = Surrogate()
    s.set_params(params, norm)
    say("mlp gradient", count)
    g, loss = s.gradient(x, t)
    s.close()
    ref_loss, ref_g = M.loss_and_grad(params.astype(np.float64), x, t, norm[:6], norm[6:])
    few = count < 1000
    assert abs(loss - ref_loss) <= (5e-3 if few else 1e-5) * ref_loss
    scale = np.abs(ref_g).max()
    assert np.max(np.abs(g - ref_g)) <= (5e-3 if few else 2e-4) * scale
