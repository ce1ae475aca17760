"""Batch normalization with the rectifier and the 2x2 max-pool behind it as a net runs them, against the operators of the
three layers: the same bits, whatever the plane's size and the net's flags."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BATCH_LIMIT = 70   # (more images than partial sums a channel has)


@pytest.mark.parametrize("flags", ["none", "all"])
@pytest.mark.parametrize("act", ["relu", "leaky_relu"])
@pytest.mark.parametrize("w,h,channels,batch", [
    (2, 2, 1, 2),        # one window
    (9, 7, 5, 3),        # a last row and column in no window
    (16, 16, 24, 37),
    (33, 40, 3, 2),      # more than 1024 elements a plane
    (5, 3, 130, BATCH_LIMIT),
])
def test_block_is_the_three_layers(T, w, h, channels, batch, act, flags):
    rng = np.random.default_rng(51)
    n, out = w * h, (w // 2) * (h // 2)
    bits = 0 if flags == "none" else T.NET_FUSE_ACT_GRAD | T.NET_GRAPH | T.NET_SAMPLE_STEP
    net = T.Net([T.L_batchnorm(channels, n), T.L_act(act), T.L_maxpool(w, h, channels, 2, 2), T.L_fc(channels * out, 3)], batch, bits)
    net.set_param(3, 0, rng.uniform(-1, 1, channels * out * 3).astype(np.float32))
    x = (rng.standard_normal((batch, channels, n)) * 2 + 0.5).astype(np.float32)
    x[0, 0, 0] = x[-1, -1, -1] = 40.0
    xd, t = T.to_device(x), T.to_device(rng.standard_normal((batch, 3)).astype(np.float32))
    buf = {k: T.DevBuf((batch, channels, n)) for k in ("y", "a", "da", "dn", "dx")}
    p, argmax = T.DevBuf((batch, channels, out)), T.DevBuf((batch, channels, out), np.int32)
    mean, var, std = (T.DevBuf((channels,)) for _ in range(3))
    pool = T.pool_desc(w, h, channels, 2, stride_w=2, stride_h=2)
    T.batchnorm_fwd(channels, n, batch, xd, mean, var, std, buf["y"])
    T.act_fwd(act, batch, channels * n, buf["y"], buf["a"])
    T.maxpool_fwd(pool, batch, buf["a"], p, argmax)

    net.train_step(None, "mse", batch, xd, t, do_update=False)
    for i, want in enumerate((buf["y"], buf["a"], p)):
        assert np.array_equal(net.layer_out(i, batch).ravel(), want.numpy().ravel()), ("forward", i)
    assert np.array_equal(net.layer_argmax(2, batch).ravel(), argmax.numpy().ravel())

    dp = T.to_device(net.layer_dx(3, batch).ravel())
    T.maxpool_bwd(pool, batch, dp, argmax, buf["da"])
    T.act_bwd(act, batch, channels * n, buf["a"], buf["da"], buf["dn"], x=buf["y"])
    T.batchnorm_bwd(channels, n, batch, buf["y"], buf["dn"], std, buf["dx"])
    if not (flags == "all" and act == "relu"):   # (folded: the gradient of relu's output stays in registers)
        assert np.array_equal(net.layer_dx(2, batch).ravel(), buf["da"].numpy().ravel())
    assert np.array_equal(net.layer_dx(1, batch).ravel(), buf["dn"].numpy().ravel())
    assert np.array_equal(net.layer_dx(0, batch).ravel(), buf["dx"].numpy().ravel())

    net.set_phase(False)                          # inference: the running averages
    net.set_param(0, 2, rng.standard_normal(channels).astype(np.float32))
    net.set_param(0, 3, rng.uniform(0.5, 2, channels).astype(np.float32))
    net.forward(batch, xd)
    T.batchnorm_fwd(channels, n, batch, xd, T.to_device(net.get_param(0, 2)), T.to_device(net.get_param(0, 3)), std, buf["y"],
                    train=False)
    T.act_fwd(act, batch, channels * n, buf["y"], buf["a"])
    T.maxpool_fwd(pool, batch, buf["a"], p, argmax)
    for i, want in enumerate((buf["y"], buf["a"], p)):
        assert np.array_equal(net.layer_out(i, batch).ravel(), want.numpy().ravel()), ("inference", i)
    net.close()
