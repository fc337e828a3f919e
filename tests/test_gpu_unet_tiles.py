"""The convolution kernels at sizes where a tile, a voxel fragment or a
channel chunk is not full, against the U-Net oracle, with
test_gpu_unet.py's tolerance (FP32 sums of exact BF16 products: 2e-5 of the
largest value), and the network at the channel counts whose decoder input
takes several chunks.
"""
import numpy as np
import pytest

from oracle import unet_oracle as U
from test_gpu_unet import _lib, _p

pytestmark = pytest.mark.gpu


# widths below, at and above a fragment (16) and a weight-gradient row (32);
# channels of one to five chunks, with and without a remainder, and of one to
# eight output tiles, among them the numbers that only 1 divides (5, 7)
@pytest.mark.parametrize("N,D,H,W,cin,cout", [
    (1, 2, 8, 6, 16, 16), (3, 1, 2, 40, 8, 24), (1, 3, 5, 16, 40, 8), (2, 1, 1, 80, 72, 40),
    (1, 5, 7, 48, 48, 48), (2, 4, 4, 17, 128, 96), (1, 1, 16, 1, 2, 3), (1, 9, 16, 64, 3, 128),
    (1, 2, 6, 48, 112, 80), (1, 3, 4, 32, 80, 112)])
def test_conv_tiles_match_oracle(N, D, H, W, cin, cout):
    L = _lib()
    rng = np.random.default_rng(cin * 17 + cout)
    x = U.bf16(rng.standard_normal((N, D, H, W, cin))).astype(np.float32)
    w = U.bf16(rng.standard_normal((cout, 27, cin)) / np.sqrt(27 * cin)).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    g = U.bf16(rng.standard_normal((N, D, H, W, cout))).astype(np.float32)
    x64, w64, g64 = (a.astype(np.float64) for a in (x, w, g))
    print(f"conv {N}x{D}x{H}x{W}, {cin} -> {cout}", flush=True)
    out = np.zeros((N, D, H, W, cout), np.float32)
    assert L.unet_conv3d(0, N, D, H, W, cin, cout, _p(x), _p(w), _p(b), 1, None, _p(out)) == 0
    ref = np.maximum(U.conv3d(x64, w64, b.astype(np.float64)), 0)
    assert np.max(np.abs(out - ref)) <= 2e-5 * np.max(np.abs(ref))
    gin = np.zeros((N, D, H, W, cin), np.float32)
    assert L.unet_conv3d(1, N, D, H, W, cin, cout, None, _p(w), None, 0, _p(g), _p(gin)) == 0
    ref = U.conv3d_bwd_data(g64, w64)
    assert np.max(np.abs(gin - ref)) <= 2e-5 * np.max(np.abs(ref))
    dw = np.zeros((cout, 27, cin), np.float32)
    assert L.unet_conv3d(2, N, D, H, W, cin, cout, _p(x), _p(w), None, 0, _p(g), _p(dw)) == 0
    ref = U.conv3d_bwd_weight(g64, x64)
    assert np.max(np.abs(dw - ref)) <= 2e-5 * np.max(np.abs(ref))


@pytest.mark.parametrize("c,in_ch,shape", [(24, 3, (1, 4, 4, 64)), (32, 2, (1, 12, 8, 128))])
def test_network_with_chunked_channels(c, in_ch, shape):
    from phasecon_amd.warmstart import UNet
    rng = np.random.default_rng(c)
    params = [(rng.standard_normal((co, 27, ci)) * np.sqrt(2.0 / (27 * ci)),
               rng.standard_normal(co) * 0.05) for ci, co, _ in U.layer_shapes(c, in_ch)]
    flat = U.flatten(params).astype(np.float32)
    net = UNet(channels=c, in_channels=in_ch)
    net.set_params(flat)
    x = rng.random(shape + (in_ch,)).astype(np.float32)
    print(f"channels {c}, {in_ch} in, {shape}", flush=True)
    y = net.forward(x)
    net.close()
    p32 = U.unflatten(flat.astype(np.float64), c, in_ch)
    t = np.zeros(shape, np.float32)
    _, _, oy = U.unet_forward_backward(p32, x, t, c, bf16_storage=True)
    # the tolerance of test_unet_gradients_match_oracle (BF16 storage points)
    assert np.max(np.abs(y - oy)) <= 1e-2 * np.max(np.abs(oy))


@pytest.mark.parametrize("c,in_ch,shape", [(24, 3, (1, 4, 4, 64)), (32, 2, (2, 8, 4, 64))])
def test_training_with_chunked_channels(c, in_ch, shape):
    """Gradients and one Adam step at the channel counts whose decoder inputs
    have 5, 9 and 12 channel tiles of 16, with the tolerances of
    test_unet_gradients_match_oracle and test_training_steps_match_oracle_adam."""
    from phasecon_amd.warmstart import UNet
    rng = np.random.default_rng(c + 1)
    params = [(rng.standard_normal((co, 27, ci)) * np.sqrt(2.0 / (27 * ci)),
               rng.standard_normal(co) * 0.05) for ci, co, _ in U.layer_shapes(c, in_ch)]
    flat = U.flatten(params).astype(np.float32)
    net = UNet(channels=c, in_channels=in_ch)
    net.set_params(flat)
    x = rng.random(shape + (in_ch,)).astype(np.float32)
    t = (x[..., 0] + 0.2 * rng.standard_normal(shape)).astype(np.float32)
    print(f"channels {c}, {in_ch} in, {shape}: gradients and a step", flush=True)
    loss, g = net.gradients(x, t)
    lr = 1e-3
    loss2 = net.train_step(x, t, lr)
    p = net.params().astype(np.float64)
    net.close()
    oloss, G, _ = U.unet_forward_backward(U.unflatten(flat.astype(np.float64), c, in_ch), x, t, c,
                                          bf16_storage=True)
    assert loss2 == loss and abs(loss - oloss) <= 1e-3 * oloss
    i = 0
    for name, (dw, db) in zip(U.LAYERS, G):
        n = dw.size + db.size
        og = U.flatten([(dw, db)])
        assert np.linalg.norm(g[i:i + n] - og) <= 3e-2 * np.linalg.norm(og), name
        i += n
    og = U.flatten(G)
    # Adam's first step: lr g / (|g| + eps)
    step = lr * og / (np.abs(og) + 1e-8)
    big = np.abs(og) > 1e-3 * np.abs(og).max()
    assert np.max(np.abs(flat - step - p)[big]) <= 0.05 * lr


def test_more_volumes_than_a_grid_axis_holds():
    """66000 volumes (a grid's second and third axis hold 65535), each equal
    to one of three: the output of every one is that of its like in a small
    batch.  The order of a voxel's sums does not depend on the batch."""
    from phasecon_amd.warmstart import UNet
    net = UNet(channels=8, seed=3)
    x = np.random.default_rng(8).random((3, 4, 4, 64)).astype(np.float32)
    print("66000 volumes of 4x4x64", flush=True)
    want = net.forward(x)
    y = net.forward(np.tile(x, (22000, 1, 1, 1))).reshape(22000, 3, 4, 4, 64)
    net.close()
    assert np.array_equal(y, np.broadcast_to(want, y.shape))
