"""A network whose buffers could not grow works again with inputs that fit."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_exact import hb, say  # noqa: F401

pytestmark = pytest.mark.gpu


def test_network_after_a_refused_gradient(hb):  # noqa: F811
    from sparkx_amd import _lib
    from sparkx_amd.surrogate import N_PARAMS
    L, net, f32 = _lib.load(), C.c_void_p(), C.c_float
    rng = np.random.default_rng(4)
    x, y = rng.standard_normal((100, 6)).astype(np.float32), rng.standard_normal(100).astype(np.float32)
    _lib.check(L.hb_mlp_create(C.byref(net), 0, 1))

    def gradient(count):
        grad = np.zeros(N_PARAMS, np.float32)
        rc = L.hb_mlp_gradient(net, _lib.ptr(x, f32), _lib.ptr(y, f32), count, _lib.ptr(grad, f32), None)
        return rc, grad

    try:
        say("gradient, refused gradient, gradient")
        rc, before = gradient(100)
        assert rc == 0 and before.any()
        assert gradient(1 << 36)[0] == -2  # HB_ENOMEM, before the inputs are read
        rc, after = gradient(100)
        assert rc == 0
        # one tile each of seven wavefronts, added by atomics in any order: a few ulp of the sums
        assert np.allclose(before, after, rtol=1e-5, atol=1e-6 * np.abs(before).max())
    finally:
        L.hb_mlp_destroy(net)
