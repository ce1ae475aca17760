"""The launch that computes dX and dW of a 5x5 convolution on 8x8 or 16x16 images together: against the oracle at the
smallest and ragged batches, and against the two gradients computed one at a time."""
import numpy as np
import pytest

from conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    # size, in_c, out_c, batch
    (8, 32, 64, 4),      # the smallest batch, every chunk its own slice
    (8, 32, 32, 37),     # a last chunk of one image, a last dX tile of one image
    (8, 64, 32, 130),    # several chunks a slice, two dX channel blocks
    (8, 96, 64, 9),
    (16, 32, 32, 4),
    (16, 32, 64, 21),    # slices that end in the middle of an image
    (16, 64, 32, 100),   # several chunks a slice
    (16, 32, 32, 131),
])
def test_matches_oracle_and_single_gradients(T, O, cfg):
    size, ic, oc, bs = cfg
    rng = np.random.default_rng(5)
    d = T.conv_desc(size, size, ic, 5, 5, oc, pad_same=True)
    x = rng.standard_normal((bs, ic * size * size)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, oc * ic * 25).astype(np.float32)
    dy = rng.standard_normal((bs, oc * size * size)).astype(np.float32)
    xd, wd, dyd = (T.to_device(a) for a in (x, w, dy))
    both = [T.DevBuf(x.shape), T.DevBuf(w.shape), T.DevBuf((oc,))]
    single = [T.DevBuf(x.shape), T.DevBuf(w.shape), T.DevBuf((oc,))]
    T.conv2d_bwd(d, bs, xd, wd, dyd, *both)
    T.conv2d_bwd(d, bs, xd, wd, dyd, single[0], None, None)
    T.conv2d_bwd(d, bs, xd, wd, dyd, None, single[1], single[2])
    want = O.conv2d_bwd(O.conv_desc(size, size, ic, 5, 5, oc, pad_same=True), x, w, dy)
    for b, s, r, name in zip(both, single, want, ("dx", "dw", "db")):
        assert_close(b.numpy().ravel(), r.ravel(), what=f"{cfg} {name}")
        assert_close(b.numpy().ravel(), s.numpy().ravel(), what=f"{cfg} {name} alone")


@pytest.mark.parametrize("flags", [0, 3])
@pytest.mark.parametrize("batch", [16, 64])
def test_first_layer_on_input_of_any_alignment(T, O, W, flags, batch):
    """The shared launch loads 16 bytes at a time. An input that lies at no multiple of 16 takes the kernels of the
    single gradients, which read filters in another layout (floats at batch 64, none at all at 16)."""
    spec = [("conv", 16, 16, 32, 5, 32, True), ("act", "tanh"), ("fc", 32 * 256, 10)]
    rng = np.random.default_rng(8)
    x = rng.standard_normal((batch, 32 * 256)).astype(np.float32)
    t = rng.uniform(-0.8, 0.8, (batch, 10)).astype(np.float32)
    room = T.to_device(np.zeros(x.size + 1, np.float32))
    xd = T.DevBuf.view(room.ptr.value + 4, x.shape, np.float32).upload(x)
    net, ref = T.Net(W.build_layers(T, spec), batch, flags), O.OracleNet(W.build_layers(O, spec), batch)
    for i, l in enumerate(spec):
        for which, n in zip((0, 1), W.layer_fans(l)[:2]):
            if n:
                a = rng.uniform(-0.02, 0.02, n).astype(np.float32)   # (tanh far from its ends)
                net.set_param(i, which, a)
                (ref.weight(i) if which == 0 else ref.bias(i))[:] = a
    opt, ropt = T.opt_desc("sgd", alpha=1e-3), O.opt_desc("sgd", alpha=1e-3)
    td = T.to_device(t)
    for _ in range(3):
        net.train_step(opt, "mse", batch, xd, td)
        ref.train_step(ropt, "mse", x, t)
        assert_close(net.layer_dx(0, batch).ravel(), ref.layer_dx(0, batch).ravel(), what="dx")
    for i in (0, 2):
        assert_close(net.get_param(i, 0), ref.weight(i), what=f"weights of layer {i}")
        assert_close(net.get_param(i, 1), ref.bias(i), what=f"bias of layer {i}")
    net.close()
