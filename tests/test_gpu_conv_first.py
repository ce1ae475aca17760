"""A net's first convolution with what leaves its kernel (activation, 2x2 max-pool, the activation behind that, and the
filters of later layers it packs along), against the operators of the layers: the same bits."""
import numpy as np
import pytest

from test_gpu_exceptional_values import check

pytestmark = pytest.mark.gpu


def conv64(x, w, b, k, stride, pad):
    batch, ci, h, wd = x.shape
    x = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    oh, ow = (h + 2 * pad - k) // stride + 1, (wd + 2 * pad - k) // stride + 1
    y = np.zeros((batch, w.shape[0], oh, ow)) + b.astype(np.float64)[None, :, None, None]
    for r in range(k):
        for s in range(k):
            part = x[:, :, r:r + stride * oh:stride, s:s + stride * ow:stride]
            y += np.tensordot(w[:, :, r, s].astype(np.float64), part, (1, 1)).transpose(1, 0, 2, 3)
    return y


@pytest.mark.parametrize("between,behind", [(None, "relu"), ("relu", None), (None, "tanh"), ("sigmoid", "relu"), ("relu", "tanh")])
@pytest.mark.parametrize("w,h,ci,k,co,batch", [
    (32, 32, 3, 5, 32, 128),    # whole tiles
    (64, 6, 1, 3, 64, 200),     # two column tiles, a last band of fewer rows
    (34, 30, 3, 5, 33, 90),     # a column tile of two, a channel tile of one
    (30, 14, 2, 3, 36, 260),
    (14, 12, 3, 5, 5, 300),
    (66, 34, 6, 4, 4, 64),      # all 96 taps
])
def test_first_convolution_is_its_layers(T, w, h, ci, k, co, batch, between, behind):
    rng = np.random.default_rng(61)
    same = k % 2 == 1
    ow, oh = (w, h) if same else (w - k + 1, h - k + 1)
    if ow % 2 or oh % 2:
        w, h, ow, oh = w + ow % 2, h + oh % 2, ow + ow % 2, oh + oh % 2
    d = T.conv_desc(w, h, ci, k, k, co, pad_same=same)
    x = rng.standard_normal((batch, ci, h, w)).astype(np.float32)
    wt = rng.uniform(-0.3, 0.3, (co, ci, k, k)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    xd, n = T.to_device(x), co * ow * oh
    y, a, p, q = T.DevBuf((batch, n)), T.DevBuf((batch, n)), T.DevBuf((batch, n // 4)), T.DevBuf((batch, n // 4))
    argmax = T.DevBuf((batch, n // 4), np.int32)
    T.profile_begin()
    T.conv2d_fwd(d, batch, xd, T.to_device(wt), T.to_device(b), y)
    assert any(r["tag"].startswith("conv_fwd_small ") for r in T.profile_end())
    ref = conv64(x, wt, b, k, 1, k // 2 if same else 0)
    bound = 2.0 ** -24 * (ci * k * k + 2) * (np.abs(x).max() * np.abs(wt).reshape(co, -1).sum(1) + np.abs(b))
    assert (np.abs(y.numpy().reshape(ref.shape) - ref) <= bound[None, :, None, None]).all()

    layers, want = [T.L_conv(w, h, ci, k, co, pad_same=same)], [y]
    if between:
        T.act_fwd(between, batch, n, y, a)
        layers, want = layers + [T.L_act(between)], want + [a]
    T.maxpool_fwd(T.pool_desc(ow, oh, co, 2, stride_w=2, stride_h=2), batch, want[-1], p, argmax)
    layers, want = layers + [T.L_maxpool(ow, oh, co, 2, 2)], want + [p]
    if behind:
        T.act_fwd(behind, batch, n // 4, p, q)
        layers, want = layers + [T.L_act(behind)], want + [q]
    net = T.Net(layers, batch, 0)
    net.set_param(0, 0, wt.ravel())
    net.set_param(0, 1, b)
    net.forward(batch, xd)
    for i, buf in enumerate(want):
        assert np.array_equal(net.layer_out(i, batch).ravel(), buf.numpy().ravel()), i
    assert np.array_equal(net.layer_argmax(len(layers) - (2 if behind else 1), batch).ravel(), argmax.numpy().ravel())
    net.close()


@pytest.mark.parametrize("convs", [1, 2, 17])    # (filters to pack: one, several, more than the 16 that a launch takes along)
def test_filters_packed_along_are_those_written_last(T, convs):
    rng = np.random.default_rng(62)
    batch, hw, c = 128, 16, 32
    layers = [T.L_conv(hw, hw, 3, 5, c, pad_same=True), T.L_act("relu")]
    layers += [T.L_conv(hw, hw, c, 3, c, pad_same=True) for _ in range(convs)]
    x, t = T.to_device(rng.standard_normal((batch, 3 * hw * hw)).astype(np.float32)), T.DevBuf((batch, c * hw * hw), zero=True)
    weights = [[rng.uniform(-0.1, 0.1, c * (3 * 25 if i == 0 else 9 * c)).astype(np.float32) for i in range(convs + 1)] for _ in (0, 1)]
    at = [0] + list(range(2, convs + 2))

    def results(net):
        out = []
        for run, jobs in ((lambda: net.forward(batch, x), convs),
                          (lambda: net.train_step(None, "mse", batch, x, t, do_update=False), 2 * convs)):
            net.clear_grads()
            T.profile_begin()
            run()
            tags = {e["tag"].split()[0] for e in T.profile_end()}
            assert "conv_fwd_small" in tags and ("conv_repack_weights" in tags) == (jobs > 16), tags
            out.append(net.layer_out(len(layers) - 1, batch).copy())
        return out + [net.layer_grad(i, 0).copy() for i in at]

    net = T.Net(layers, batch, T.NET_FUSE_ACT_GRAD)
    views = [T.DevBuf.view(T.lib().tdh_net_param(net.h, i, 0), (net.param_size(i, 0),)) for i in at]   # (never trusted again)
    got = []
    for ws in weights:
        for view, v in zip(views, ws):
            view.upload(v)
        got.append(results(net))
    net.close()
    for ws, have in zip(weights, got):
        fresh = T.Net(layers, batch, T.NET_FUSE_ACT_GRAD)
        for i, v in zip(at, ws):
            fresh.set_param(i, 0, v)
        for i, (a, b) in enumerate(zip(have, results(fresh))):
            assert np.array_equal(a, b), i
        fresh.close()


@pytest.mark.parametrize("w,h,ci,k,co,batch", [
    (32, 32, 3, 5, 32, 128),    # 75 taps of 80
    (28, 28, 1, 5, 33, 256),    # 25 of 32
    (30, 20, 3, 3, 20, 160),    # 27 of 32
    (40, 24, 6, 4, 16, 100),    # all 96
])
def test_what_fills_up_the_taps_is_no_part_of_a_sum(T, w, h, ci, k, co, batch):
    """Infinities and NaN under the first tap of the first channel, whose place the taps that fill up a block of 16 take."""
    rng = np.random.default_rng(63)
    same = k % 2 == 1
    ow, oh = (w, h) if same else (w - k + 1, h - k + 1)
    ow, oh = ow - ow % 2, oh - oh % 2
    w, h = (ow, oh) if same else (ow + k - 1, oh + k - 1)
    d = T.conv_desc(w, h, ci, k, k, co, pad_same=same)
    x = rng.standard_normal((batch, ci, h, w)).astype(np.float32)
    for i, v in enumerate([np.inf, -np.inf, np.nan, np.inf, 3e37]):
        x[rng.integers(batch), 0, rng.integers(h), rng.integers(w)] = v
        x[i, 0, 0, 0] = v
    wt = rng.uniform(0.1, 0.3, (co, ci, k, k)).astype(np.float32) * rng.choice([-1, 1], (co, ci, k, k)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    xd, n = T.to_device(x), co * ow * oh
    y, p, argmax = T.DevBuf((batch, n)), T.DevBuf((batch, n // 4)), T.DevBuf((batch, n // 4), np.int32)
    T.profile_begin()
    T.conv2d_fwd(d, batch, xd, T.to_device(wt), T.to_device(b), y)
    assert any(r["tag"].startswith("conv_fwd_small ") for r in T.profile_end())
    with np.errstate(invalid="ignore"):
        check(y.numpy(), conv64(x, wt, b, k, 1, k // 2 if same else 0), "y")
    T.maxpool_fwd(T.pool_desc(ow, oh, co, 2, stride_w=2, stride_h=2), batch, y, p, argmax)
    net = T.Net([T.L_conv(w, h, ci, k, co, pad_same=same), T.L_maxpool(ow, oh, co, 2, 2)], batch, 0)
    net.set_param(0, 0, wt.ravel())
    net.set_param(0, 1, b)
    net.forward(batch, xd)
    assert np.array_equal(net.layer_out(0, batch).ravel(), y.numpy().ravel(), equal_nan=True)
    assert np.array_equal(net.layer_out(1, batch).ravel(), p.numpy().ravel(), equal_nan=True)
    assert np.array_equal(net.layer_argmax(1, batch).ravel(), argmax.numpy().ravel())
    net.close()


@pytest.mark.parametrize("co", [3, 33])
def test_planes_of_more_than_a_descriptor(T, co):
    """2^25 pixels of 32 channels are 4 GiB, more than one buffer descriptor reaches."""
    rng = np.random.default_rng(64)
    w, h, k = 2050, 16500, 3
    assert w * h > 1 << 25
    x = rng.standard_normal((1, 1, h, w)).astype(np.float32)
    wt = rng.uniform(-0.3, 0.3, (co, 1, k, k)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    y = T.DevBuf((co * h * w,))
    T.profile_begin()
    T.conv2d_fwd(T.conv_desc(w, h, 1, k, k, co, pad_same=True), 1, T.to_device(x), T.to_device(wt), T.to_device(b), y)
    assert any(r["tag"].startswith("conv_fwd_small ") for r in T.profile_end())
    bound = 2.0 ** -24 * (k * k + 2) * (np.abs(x).max() * np.abs(wt).reshape(co, -1).sum(1) + np.abs(b))
    for row in (1, 8191, h - 2):
        want = conv64(x[:, :, row - 1:row + 2], wt, b, k, 1, 1)[0, :, 1]
        for c in range(co):
            got = T.DevBuf.view(y.ptr.value + 4 * (c * h + row) * w, (w,)).numpy()
            assert (np.abs(got - want[c]) <= bound[c]).all(), (row, c)


def test_more_work_items_than_a_grid_has_in_one_direction(T):
    """65535 images of 513 blocks of channels, a workgroup of two waves each: more than 2^32 work-items."""
    rng = np.random.default_rng(65)
    k, co, batch = 3, 32 * 513, 65535
    x = rng.standard_normal((batch, 1, k, k)).astype(np.float32)
    wt = rng.uniform(-0.3, 0.3, (co, 1, k, k)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    y = T.DevBuf((batch * co,))
    T.profile_begin()
    T.conv2d_fwd(T.conv_desc(k, k, 1, k, k, co), batch, T.to_device(x), T.to_device(wt), T.to_device(b), y)
    assert any(r["tag"].startswith("conv_fwd_small ") for r in T.profile_end())
    bound = 2.0 ** -24 * (k * k + 2) * (np.abs(x).max() * np.abs(wt).reshape(co, -1).sum(1) + np.abs(b))
    for i in (0, 1, 4095, 32768, 65533, 65534):
        got = T.DevBuf.view(y.ptr.value + 4 * i * co, (co,)).numpy()
        want = wt.reshape(co, -1).astype(np.float64) @ x[i].ravel().astype(np.float64) + b
        assert (np.abs(got - want) <= bound).all(), i


@pytest.mark.parametrize("w,h,ci,k,co,batch,same", [
    (128, 9, 3, 3, 17, 4, True),     # rows of 128, the last band of one row, a last chunk of one channel
    (20, 21, 4, 3, 8, 9, True),
    (26, 19, 2, 3, 5, 9, False),     # rows of 24 outputs, two in front of the first that is read
    (40, 13, 1, 5, 9, 6, True),
    (44, 30, 4, 5, 30, 3, False),    # rows of 40 outputs from the first one on
    (200, 31, 3, 3, 9, 12, True),    # a band of one row
])
def test_dx_of_words_is_that_of_elements(T, w, h, ci, k, co, batch, same):
    """dX reads rows of a multiple of four outputs by words where they are aligned, else by elements: the same bits, and the
    same as a correlation in 64 bits (the error of a sum of k * k * co products)."""
    rng = np.random.default_rng(5)
    ow, oh = (w, h) if same else (w - k + 1, h - k + 1)
    d = T.conv_desc(w, h, ci, k, k, co, pad_same=same)
    wt = rng.uniform(-0.3, 0.3, (co, ci, k, k)).astype(np.float32)
    dy = rng.standard_normal((batch, co, oh, ow)).astype(np.float32)
    moved = T.DevBuf((dy.size + 1,))
    moved.upload(np.concatenate([[0], dy.ravel()]).astype(np.float32))
    x, got = T.to_device(rng.standard_normal((batch, ci, h, w)).astype(np.float32)), []
    for g in (T.to_device(dy), T.DevBuf.view(moved.ptr.value + 4, dy.shape)):
        dx = T.DevBuf((batch, ci, h, w))
        T.profile_begin()
        T.conv2d_bwd(d, batch, x, T.to_device(wt), g, dx, T.DevBuf(wt.shape), T.DevBuf((co,)))
        tags = [r["tag"].split()[0] for r in T.profile_end()]
        assert "conv_dx_small_cin" in tags, tags
        got.append(dx.numpy())
    assert np.array_equal(*got)
    p = k // 2 if same else 0
    want, size = np.zeros((2, batch, ci, h + 2 * p, w + 2 * p))
    dy, wt = dy.astype(np.float64), wt.astype(np.float64)
    for ky in range(k):
        for kx in range(k):
            at = (slice(None), slice(None), slice(ky, ky + oh), slice(kx, kx + ow))
            want[at] += np.einsum("bohw,oc->bchw", dy, wt[:, :, ky, kx])
            size[at] += np.einsum("bohw,oc->bchw", np.abs(dy), np.abs(wt[:, :, ky, kx]))
    inner = (slice(None), slice(None), slice(p, p + h), slice(p, p + w))
    assert np.all(np.abs(got[0] - want[inner]) <= 2.0**-24 * (k * k * co + 2) * size[inner])
