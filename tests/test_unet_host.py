"""The network's host side against a stand-in for the HIP runtime
(hip_stub.py): what a failed allocation leaves behind, and the grids of
launches over many volumes."""
import os

import numpy as np
import pytest

import hip_stub

pytestmark = pytest.mark.skipif(not os.path.exists(hip_stub.HIPCC), reason="no hipcc")


@pytest.fixture
def L(monkeypatch):
    return hip_stub.use(monkeypatch)


@pytest.mark.parametrize("after", [0, 1, 7, 20, 29])
def test_a_shape_whose_buffers_failed_is_not_kept(L, after):
    """Whichever of a new shape's buffers fails, the next call of the same
    shape allocates them all again and never launches on the ones that are
    missing or freed."""
    from phasecon_amd.warmstart import UNet
    live0 = L.stub_live()
    net = UNet(channels=8)
    small, large = (np.zeros(s, np.float32) for s in ((1, 4, 4, 64), (2, 8, 8, 64)))
    net.forward(small)
    live = L.stub_live()
    L.stub_fail_malloc(after)
    n = L.stub_launches()
    for _ in range(2):                          # the second: still no memory
        with pytest.raises(RuntimeError):
            net.forward(large)
    assert L.stub_launches() == n
    L.stub_fail_malloc(-1)
    before = L.stub_mallocs()
    net.forward(large)
    assert L.stub_live() == live                # a whole set, and nothing lost
    assert L.stub_mallocs() - before > after
    net.forward(small)
    net.close()
    assert L.stub_live() == live0


@pytest.mark.parametrize("shape", [(66000, 4, 4, 64), (1, 4, 70000 * 8, 64)])
def test_grids_of_many_tiles(L, shape):
    """Volumes, and tiles along y, beyond what a grid's second and third axis
    hold (65535)."""
    from phasecon_amd.warmstart import UNet
    net = UNet(channels=8)
    x = np.zeros(shape, np.float32)
    L.stub_clear_log()
    net.forward(x)
    net.close()
    runs = hip_stub.launches(L)
    assert sum("k_conv" in r[0] for r in runs) > 11
    for name, gx, gy, gz, threads in runs:
        assert gy <= 65535 and gz <= 65535 and gx * threads < 1 << 32, name
