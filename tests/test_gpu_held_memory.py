"""Device memory kept after an exact search is given back when any allocation of the library
fails, whichever part of it allocates, and on request."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_exact import hb, say  # noqa: F401
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu

MTX = b"%%MatrixMarket matrix coordinate pattern symmetric\n3 3 2\n2 1\n3 2\n"


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _hold(hb):  # noqa: F811
    """An exact search over sources enough for a block of more than 512 MiB; returns what is
    free with the block kept."""
    from sparkx_amd.exact import ExactHarmonicCentrality
    g = hb.Graph.erdos_renyi(1 << 19, 1 << 19, seed=3)
    ExactHarmonicCentrality(g, True, sources=(0, 2048))
    return _free_bytes()


def _network():
    """A gradient over more samples than the device can hold: refused before they are read."""
    from sparkx_amd import _lib
    from sparkx_amd.surrogate import N_PARAMS
    L, net = _lib.load(), C.c_void_p()
    _lib.check(L.hb_mlp_create(C.byref(net), 0, 1))
    x, grad = np.zeros(6, np.float32), np.zeros(N_PARAMS, np.float32)
    f32 = C.c_float
    rc = L.hb_mlp_gradient(net, _lib.ptr(x, f32), _lib.ptr(x, f32), 1 << 36, _lib.ptr(grad, f32), None)
    L.hb_mlp_destroy(net)
    return rc


def _text():
    """A MatrixMarket text said to be longer than the device's memory."""
    from sparkx_amd import _lib
    L, ctx = _lib.load(), C.c_void_p()
    _lib.check(L.hb_create(C.byref(ctx), 0))
    rc = L.hb_stage_mtx(ctx, MTX, 1 << 40, None)
    L.hb_destroy(ctx)
    return rc


@pytest.mark.parametrize("allocate", [_network, _text])
def test_failed_allocation_gives_back_what_is_held(hb, allocate):  # noqa: F811
    held = _hold(hb)
    say("held", allocate.__name__, held)
    assert allocate() == -2  # HB_ENOMEM
    assert _free_bytes() >= held + (512 << 20)
    # the failure is reported once, by the call that failed
    with hb.HyperBall(hb.Graph.erdos_renyi(1000, 4000, seed=1), 6) as h:
        assert h.get_iters() > 1


def test_release_on_request(hb):  # noqa: F811
    held = _hold(hb)
    say("held", held)
    hb.release_memory()
    assert _free_bytes() >= held + (512 << 20)
    hb.release_memory()  # nothing left: no effect
    assert _hold(hb) <= held + (64 << 20)
