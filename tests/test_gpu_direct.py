"""The forward kernels for layers of a few small tiles: convolutions against the oracle at the edges of their 16 x 16
tiles and of their blocks of 16 indices, and nets (pool, activations and softmax in the layer's launch) at inference."""
import numpy as np
import pytest

from conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    # in_w, in_h, in_c, k, out_c, same, stride, dilation, batch
    (5, 5, 1, 5, 1, False, 1, 1, 1),         # one pixel, one channel
    (9, 7, 3, 3, 16, True, 1, 1, 1),         # 27 indices: W read float by float
    (8, 8, 16, 1, 17, False, 1, 1, 3),       # one block of indices, a second tile of one channel
    (13, 11, 4, 4, 20, True, 1, 1, 2),       # a last tile of 14 pixels
    (12, 12, 32, 5, 33, True, 1, 1, 2),      # 800 indices: sixteen waves
    (10, 9, 24, 3, 8, False, 1, 1, 4),       # 216 indices: four waves
    (11, 10, 40, 3, 12, False, 2, 1, 3),     # eight waves, strided
    (14, 13, 6, 3, 10, False, 1, 2, 2),      # dilated
    (4, 4, 2048, 1, 16, False, 1, 1, 1),     # the longest reduction
    (32, 30, 5, 7, 64, True, 1, 1, 2),
])
def test_conv_matches_oracle(T, O, cfg):
    iw, ih, ic, k, oc, same, st, dil, bs = cfg
    rng = np.random.default_rng(11)
    kw = dict(pad_same=same, w_stride=st, h_stride=st, w_dilation=dil, h_dilation=dil)
    d = T.conv_desc(iw, ih, ic, k, k, oc, **kw)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic * ih * iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, oc * ic * k * k).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    y = T.DevBuf((bs, oc * oh * ow))
    T.conv2d_fwd(d, bs, T.to_device(x), T.to_device(w), T.to_device(b), y)
    assert_close(y.numpy().ravel(), O.conv2d_fwd(O.conv_desc(iw, ih, ic, k, k, oc, **kw), x, w, b).ravel(), what=str(cfg))


@pytest.mark.parametrize("batch", [1, 3, 17])
@pytest.mark.parametrize("flags", [0, 3])
@pytest.mark.parametrize("spec", [
    [("conv", 12, 12, 3, 5, 20, True), ("maxpool", 12, 12, 20, 2), ("act", "tanh"),
     ("conv", 6, 6, 20, 3, 18, True), ("act", "relu"), ("maxpool", 6, 6, 18, 2), ("fc", 162, 30), ("act", "sigmoid"),
     ("fc", 30, 16), ("act", "softmax")],
    [("conv", 10, 8, 2, 3, 5, False), ("act", "tanh"), ("maxpool", 8, 6, 5, 2), ("fc", 60, 17), ("act", "softmax")],
    [("fc", 2048, 40), ("act", "relu"), ("fc", 40, 1), ("act", "softmax")],
])
def test_inference_matches_oracle(T, O, W, spec, flags, batch):
    rng = np.random.default_rng(7)
    net, ref = T.Net(W.build_layers(T, spec), batch, flags), O.OracleNet(W.build_layers(O, spec), batch)
    for i, l in enumerate(spec):
        nw, nb, _, _ = W.layer_fans(l)
        for which, n in ((0, nw), (1, nb)):
            if n:
                a = rng.uniform(-0.2, 0.2, n).astype(np.float32)
                net.set_param(i, which, a)
                (ref.weight(i) if which == 0 else ref.bias(i))[:] = a
    x = rng.standard_normal((batch, net.in_size())).astype(np.float32)
    net.forward(batch, T.to_device(x))
    ref.forward(x)
    for i in range(len(spec)):
        assert_close(net.layer_out(i, batch).ravel(), ref.layer_out(i, batch).ravel(), what=f"layer {i}")
    net.close()


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("cfg", [
    # in_w, in_h, in_c, k, out_c, same, stride, batch
    (5, 5, 1, 5, 1, False, 1, 1),         # one output pixel
    (9, 7, 3, 3, 16, True, 1, 1),         # db in a tile of its own columns' end: 27 + 1
    (9, 8, 5, 3, 17, True, 1, 2),         # 45 + 1 columns, rows that are no multiple of four
    (8, 8, 16, 1, 20, False, 1, 3),       # 16 columns: db alone in the second tile
    (12, 12, 32, 5, 33, True, 1, 2),      # 825 indices of dX: sixteen waves
    (16, 16, 8, 3, 24, True, 1, 8),       # 2048 pixels
    (11, 10, 20, 3, 12, False, 2, 3),     # strided, rows that no window reaches
    (13, 12, 6, 4, 10, True, 3, 2),       # stride 3, window of 4
    (12, 9, 4, 1, 9, False, 2, 2),        # stride larger than the window
    # too many pixels for that launch: the bias gradient is a column of the weight gradient's product
    (27, 25, 5, 3, 9, False, 2, 17),      # 2856 pixels, 46 columns
    (31, 29, 1, 1, 5, True, 1, 3),        # one weight and the bias
    (25, 26, 7, 3, 40, True, 1, 4),       # 64 columns with the bias gradient's
    (25, 26, 32, 1, 6, True, 1, 4),       # 32 columns without it: it stays a launch of its own
])
def test_conv_gradients_match_oracle(T, O, cfg, accumulate):
    iw, ih, ic, k, oc, same, st, bs = cfg
    rng = np.random.default_rng(12)
    kw = dict(pad_same=same, w_stride=st, h_stride=st)
    d = T.conv_desc(iw, ih, ic, k, k, oc, **kw)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic * ih * iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, oc * ic * k * k).astype(np.float32)
    dy = rng.standard_normal((bs, oc * oh * ow)).astype(np.float32)
    start = [rng.standard_normal(n).astype(np.float32) if accumulate else np.full(n, 7, np.float32) for n in (w.size, oc)]
    dx, dw, db = T.DevBuf(x.shape), T.to_device(start[0]), T.to_device(start[1])
    T.conv2d_bwd(d, bs, T.to_device(x), T.to_device(w), T.to_device(dy), dx, dw, db, accumulate=accumulate)
    want = O.conv2d_bwd(O.conv_desc(iw, ih, ic, k, k, oc, **kw), x, w, dy)
    base = [np.zeros(1), *(start if accumulate else (np.zeros(1), np.zeros(1)))]
    for g, r, b, name in zip((dx, dw, db), want, base, ("dx", "dw", "db")):
        assert_close(g.numpy().ravel(), r.ravel() + b, what=f"{cfg} {name}")
