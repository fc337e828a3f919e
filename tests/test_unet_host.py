"""The network's host side against a stand-in for the HIP runtime
(hip_stub.py): what a failed allocation leaves behind."""
import ctypes as C
import os

import numpy as np
import pytest

import hip_stub

pytestmark = pytest.mark.skipif(not os.path.exists(hip_stub.HIPCC), reason="no hipcc")


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    return hip_stub.build("unet_hip", str(tmp_path_factory.mktemp("unet")))


def _p(a):
    return a.ctypes.data_as(C.c_void_p)


def _net(L, channels=8):
    h = C.c_void_p()
    assert L.unet_create(C.byref(h), channels, 1, 0) == 0
    return h


def _forward(L, h, shape):
    x, y = np.zeros(shape, np.float32), np.empty(shape, np.float32)
    return L.unet_forward(h, *shape, _p(x), _p(y))


@pytest.mark.parametrize("after", [0, 1, 7, 20, 29])
def test_a_shape_whose_buffers_failed_is_not_kept(L, after):
    """Whichever of a new shape's buffers fails, the next call of the same
    shape allocates them all again and never launches on the ones that are
    missing or freed."""
    h = _net(L)
    small, large = (1, 4, 4, 64), (2, 8, 8, 64)
    assert _forward(L, h, small) == 0
    live = L.stub_live()
    L.stub_fail_malloc(after)
    assert _forward(L, h, large) == -1
    n = L.stub_launches()
    assert _forward(L, h, large) == -1          # still no memory
    assert L.stub_launches() == n
    L.stub_fail_malloc(-1)
    before = L.stub_mallocs()
    assert _forward(L, h, large) == 0
    assert L.stub_live() == live                # a whole set, and nothing lost
    assert L.stub_mallocs() - before > after
    assert _forward(L, h, small) == 0
    L.unet_destroy(h)
    assert L.stub_live() == 0
