"""A 2x2 max-pool that leaves the stride-1 convolution's kernel in rows of 32 and 64 pixels, where a wave's blocks are pairs of
rows: bit for bit what the pool's own kernel makes of the same convolution."""
import numpy as np
import pytest

from conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["train", "forward"])
@pytest.mark.parametrize("act", [None, "relu", "tanh"])
@pytest.mark.parametrize("behind", [None, "relu"])
@pytest.mark.parametrize("width,height,in_c,out_c,window,batch", [
    (24, 22, 32, 40, 3, 130),    # rows of 32, three quarters of them used; a last tile of six rows
    (34, 18, 11, 64, 5, 45),     # two tiles a row, the second two pixels wide; a window of five
    (48, 46, 32, 64, 3, 33),     # rows of 64
    (66, 6, 30, 33, 3, 98),      # a tile of four rows, half of the last one; one channel in a second block
    (130, 4, 31, 70, 3, 65),     # an image of one tile's rows
    (64, 2, 32, 48, 3, 771),     # fewer rows than a tile: two images in it, the last one alone
    (32, 34, 32, 24, 3, 130),    # 32 channels or fewer: tiles of 512 pixels
    (70, 66, 32, 32, 3, 22),
])
def test_pool_of_rows_as_its_own_kernel(T, W, width, height, in_c, out_c, window, batch, act, behind, form):
    spec = [("conv", width, height, in_c, window, out_c, True)] + ([("act", act)] if act else [])
    spec += [("maxpool", width, height, out_c, 2)] + ([("act", behind)] if behind else [])
    rng = np.random.default_rng(7)
    w = rng.uniform(-0.3, 0.3, out_c * in_c * window * window).astype(np.float32)
    b = np.linspace(-0.2, 0.2, out_c, dtype=np.float32)
    x = T.to_device(rng.standard_normal((batch, width * height * in_c)).astype(np.float32))
    # (a train step of a fusing net, as VGG's: with an activation behind it the convolution's own output stays unwritten)
    fusing = form == "train" and (not act or behind)
    net = T.Net(W.build_layers(T, spec), batch, T.NET_FUSE_ACT_GRAD if fusing else 0)
    net.set_param(0, 0, w)
    net.set_param(0, 1, b)
    pool = 2 if act else 1
    y = T.DevBuf((batch, width * height * out_c))
    T.conv2d_fwd(T.conv_desc(width, height, in_c, window, window, out_c, pad_same=True), batch, x, T.to_device(w), T.to_device(b), y)
    t = T.DevBuf((batch, net.layer_out_size(len(spec) - 1)), zero=True)
    T.profile_begin()
    if form == "train":
        net.train_step(None, "mse", batch, x, t, do_update=False)
        assert net.out_written(0) == (not act or not fusing)
        if net.out_written(0):
            assert_close(net.layer_out(0, batch), y.numpy())
    else:
        net.forward(batch, x)
        assert np.array_equal(net.layer_out(0, batch), y.numpy())
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    # (inference takes the three-part kernel, which has the pool in rows of 32 only)
    want = "conv_fwd_s1_pool" if form == "train" else "conv_fwd_x3_pool" if width < 48 else "conv_fwd_x3"
    assert want in tags and any(tag.startswith("maxpool_fwd") for tag in tags) == (want == "conv_fwd_x3"), tags
    read = net.layer_out(pool - 1, batch)
    if not net.out_written(0):
        assert_close(read, np.maximum(y.numpy(), 0) if act == "relu" else np.tanh(y.numpy()))
    elif act == "relu":
        assert np.array_equal(read, np.maximum(net.layer_out(0, batch), 0))
    planes = read.reshape(batch, out_c, height // 2, 2, width // 2, 2).transpose(0, 1, 2, 4, 3, 5).reshape(batch, out_c, -1, 4)
    first  = planes.argmax(-1)
    want   = np.take_along_axis(planes, first[..., None], -1)[..., 0]
    assert np.array_equal(net.layer_out(pool, batch).ravel(), want.ravel())
    if behind:
        assert np.array_equal(net.layer_out(pool + 1, batch).ravel(), np.maximum(want, 0).ravel())
    at = np.arange(want.shape[-1])
    top = 2 * (at // (width // 2)) * width + 2 * (at % (width // 2))
    record = (np.arange(out_c) * height * width)[None, :, None] + top[None, None, :] + (first >> 1) * width + (first & 1)
    assert np.array_equal(net.layer_argmax(pool, batch).ravel(), record.ravel())
    net.close()


@pytest.mark.parametrize("window", [3, 5])
def test_rows_of_64_take_no_longer_than_rows_of_32(T, W, window):
    """A train step's forward pass of 32 channels or fewer, in tiles of 512 pixels: as many products in rows of either length.
    (With the blocks of the wider rows in another order the kernel's registers went to memory: 1.13 and 1.27 times; else 1.00 and 1.02.)"""
    us = {}
    for width, batch in ((32, 256), (64, 64)):
        layers = W.build_layers(T, [("conv", width, width, 32, window, 32, True)])
        net = T.Net(layers, batch, 0)
        for i, which, n in net.params():
            net.set_param(i, which, np.linspace(-0.1, 0.1, n, dtype=np.float32))
        x = T.to_device(np.linspace(-1, 1, batch * net.in_size(), dtype=np.float32).reshape(batch, -1))
        t = T.DevBuf((batch, net.layer_out_size(0)), zero=True)
        net.train_step(None, "mse", batch, x, t, do_update=False)
        best = float("inf")
        for _ in range(5):
            T.profile_begin()
            for _ in range(10):
                net.train_step(None, "mse", batch, x, t, do_update=False)
            best = min([best] + [e["avg_us"] for e in T.profile_end() if e["tag"].startswith("conv_fwd_s1")])
        us[width] = best
        net.close()
    print(us)
    assert us[64] < 1.08 * us[32], us
