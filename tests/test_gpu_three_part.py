"""The convolution and fully-connected kernels on three-part bf16 operands: against the oracle at the edges of their tiles,
and against float64, from which they may be no further than a sum in fp32."""
import numpy as np
import pytest

from conftest import assert_close

pytestmark = pytest.mark.gpu


def run(T, cfg, rng, spread=0.0, scale=(0, 0, 0)):
    iw, ih, ic, k, oc, same, bs = cfg
    d = T.conv_desc(iw, ih, ic, k, k, oc, pad_same=same)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic * ih * iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, oc * ic * k * k).astype(np.float32)
    dy = rng.standard_normal((bs, oc * oh * ow)).astype(np.float32)
    if spread:
        x *= np.exp(spread * rng.standard_normal(x.shape)).astype(np.float32)
    for a, e in zip((x, w, dy), scale):
        a *= np.float32(2.0 ** e)
    b = rng.standard_normal(oc).astype(np.float32) * np.float32(2.0 ** (scale[0] + scale[1]))
    xd, wd, dyd, bd = (T.to_device(a) for a in (x, w, dy, b))
    y, dx, dw, db = T.DevBuf(dy.shape), T.DevBuf(x.shape), T.DevBuf(w.shape), T.DevBuf((oc,))
    T.conv2d_fwd(d, bs, xd, wd, bd, y)
    T.conv2d_bwd(d, bs, xd, wd, dyd, dx, dw, db)
    return (x, w, b, dy), [a.numpy() for a in (y, dx, dw, db)]


@pytest.mark.parametrize("cfg", [
    # in_w, in_h, in_c, k, out_c, same, batch
    (64, 12, 16, 3, 64, True, 86),      # one chunk of channels
    (66, 17, 33, 3, 65, True, 26),      # channels past a chunk and a tile, a second column tile, scalar loads
    (50, 11, 40, 3, 24, False, 37),     # no padding, fewer than 32 channels in dX
    (17, 33, 48, 3, 96, True, 33),      # tiles of 16 columns, ragged rows
    (30, 30, 64, 3, 40, False, 20),     # tiles of 32 columns
    (8, 8, 32, 5, 64, True, 600),       # several images a tile
    (16, 16, 32, 5, 20, True, 300),     # 5x5
    (53, 50, 20, 5, 40, True, 7),       # 5x5, scalar loads: dW by filter-row groups, one of them half empty
    (49, 50, 34, 5, 33, False, 6),
    (40, 40, 50, 1, 70, True, 12),      # 1x1
    (36, 30, 20, 7, 40, True, 12),      # 7x7
    (128, 4, 64, 3, 64, True, 65),      # images of fewer rows than a slice warms up
])
def test_matches_oracle(T, O, cfg):
    iw, ih, ic, k, oc, same, bs = cfg
    (x, w, b, dy), got = run(T, cfg, np.random.default_rng(3))
    do = O.conv_desc(iw, ih, ic, k, k, oc, pad_same=same)
    want = [O.conv2d_fwd(do, x, w, b), *O.conv2d_bwd(do, x, w, dy)]
    for g, r, name in zip(got, want, ("y", "dx", "dw", "db")):
        assert_close(g.ravel(), r.ravel(), what=f"{cfg} {name}")


@pytest.mark.parametrize("cfg", [
    # (of the list above, the ones that have too few tiles there for the three-part kernels in both directions)
    (50, 11, 40, 3, 24, False, 130),
    (30, 30, 64, 3, 40, False, 70),
    (53, 50, 20, 5, 40, True, 20),
    (49, 50, 34, 5, 33, False, 24),
    (40, 40, 50, 1, 70, True, 26),
    (36, 30, 20, 7, 40, True, 33),
])
def test_every_window_against_float64(T, cfg):
    import torch
    iw, ih, ic, k, oc, same, bs = cfg
    T.profile_begin()
    (x, w, b, dy), got = run(T, cfg, np.random.default_rng(3))
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert {"conv_fwd_x3", "conv_dx_x3"} <= tags, tags
    xt = torch.from_numpy(x).double().reshape(bs, ic, ih, iw).requires_grad_()
    wt = torch.from_numpy(w).double().reshape(oc, ic, k, k).requires_grad_()
    y = torch.nn.functional.conv2d(xt, wt, torch.from_numpy(b).double(), padding=k // 2 if same else 0)
    y.backward(torch.from_numpy(dy).double().reshape(y.shape))
    for g, r, name in zip(got, (y, xt.grad, wt.grad), ("y", "dx", "dw")):
        assert_close(g.ravel(), r.detach().numpy().ravel(), what=f"{cfg} {name}")


@pytest.mark.parametrize("cfg", [
    # in, out, batch
    (4096, 1024, 64),      # tiles of 64 rows
    (1028, 1012, 260),     # ragged on every side, a last step of four indices
    (2048, 64, 512),       # tiles of 64 columns
    (16384, 68, 132),      # a reduction of two steps and four indices
    # (of the first three, forward and dX are left to other kernels: too few tiles)
    (8192, 2048, 64),      # tiles of 64 rows
    (1028, 1012, 520),     # ragged on every side
    (4096, 64, 2048),      # tiles of 64 columns, dX with the shortest reduction
])
def test_fc_matches_oracle(T, O, W, cfg):
    """dX as an operator, the forward product as a net's inference."""
    ni, no, bs = cfg
    rng = np.random.default_rng(6)
    x = rng.standard_normal((bs, ni)).astype(np.float32)
    w = rng.uniform(-0.2, 0.2, ni * no).astype(np.float32)
    b = rng.standard_normal(no).astype(np.float32)
    dy = rng.standard_normal((bs, no)).astype(np.float32)
    xd, dx = T.to_device(x), T.DevBuf(x.shape)
    T.profile_begin()
    T.fc_bwd(ni, no, True, bs, xd, T.to_device(w), T.to_device(dy), dx, None, None)
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert "fc_dx_x3" in tags or cfg in ((4096, 1024, 64), (1028, 1012, 260), (2048, 64, 512)), tags
    assert_close(dx.numpy(), O.fc_bwd(x, w, dy)[0], what=f"{cfg} dx")
    want = O.fc_fwd(x, w, b)
    for flags, act in ((0, False), (T.NET_FUSE_ACT_GRAD, True)):
        spec = [("fc", ni, no)] + ([("act", "relu")] if act else [])
        net = T.Net(W.build_layers(T, spec), bs, flags)
        net.set_param(0, 0, w); net.set_param(0, 1, b)
        net.forward(bs, xd)
        assert_close(net.layer_out(0, bs), want, what=f"{cfg} y")
        if act:
            assert_close(net.layer_out(1, bs), np.maximum(want, 0), what=f"{cfg} relu")
        net.close()


@pytest.mark.parametrize("spread, scale", [
    (0.0, (0, 0, 0)), (3.0, (0, 0, 0)),
    # powers of two of x, w and dy: operands whose lowest bits are far below the smallest normal bf16
    (0.0, (-116, 0, 0)), (0.0, (0, -116, 0)), (0.0, (0, 0, -116)), (0.0, (-118, 30, 30)), (0.0, (-60, -50, -58)),
])
def test_no_further_from_float64_than_fp32_sums(T, spread, scale):
    import torch
    cfg = (64, 64, 32, 3, 64, True, 16)
    iw, ih, ic, k, oc, _, bs = cfg
    (x, w, b, dy), got = run(T, cfg, np.random.default_rng(4), spread, scale)
    xt = torch.from_numpy(x).double().reshape(bs, ic, ih, iw).requires_grad_()
    wt = torch.from_numpy(w).double().reshape(oc, ic, k, k).requires_grad_()
    y = torch.nn.functional.conv2d(xt, wt, torch.from_numpy(b).double(), padding=1)
    y.backward(torch.from_numpy(dy).double().reshape(y.shape))
    for g, r, name in zip(got, (y, xt.grad, wt.grad), ("y", "dx", "dw")):
        r = r.detach().numpy().ravel()
        e = g.ravel().astype(np.float64) - r
        # (a sum of n products rounded after each: sqrt(n) half-ulps and more; the fp32 kernels
        # measure 2.2e-7 to 3.0e-7 here)
        assert np.linalg.norm(e) <= 2.0e-7 * np.linalg.norm(r), (name, np.linalg.norm(e) / np.linalg.norm(r))
        assert abs(e.mean()) <= 2e-8 * np.sqrt(np.mean(r * r)), (name, e.mean())


@pytest.mark.parametrize("scale", [(-120, 0), (0, -120), (-60, -52)])
def test_fc_of_tiny_operands(T, W, scale):
    ni, no, bs = 1024, 1024, 512
    rng = np.random.default_rng(16)
    x = rng.standard_normal((bs, ni)).astype(np.float32) * np.float32(2.0 ** scale[0])
    w = rng.uniform(-0.2, 0.2, ni * no).astype(np.float32) * np.float32(2.0 ** scale[1])
    net = T.Net(W.build_layers(T, [("fc", ni, no)]), bs, 0)
    net.set_param(0, 0, w)
    net.set_param(0, 1, np.zeros(no, np.float32))
    xd, wd, dx = T.to_device(x), T.to_device(w), T.DevBuf(x.shape)
    net.forward(bs, xd)
    T.fc_bwd(ni, no, True, bs, xd, wd, xd, dx, None, None)   # (square: x stands for dy)
    w64 = w.astype(np.float64).reshape(ni, no)
    for got, want, name in ((net.layer_out(0, bs), x @ w64, "y"), (dx.numpy(), x @ w64.T, "dx")):
        # (a sum of 1024 products rounded after each: sqrt(1024) half-ulps, 9.5e-7)
        assert np.linalg.norm(got - want) <= 5.0e-7 * np.linalg.norm(want), name
    net.close()


@pytest.mark.parametrize("batch", [4, 32, 64])
def test_convolution_operator_and_inference_are_one_product(T, W, batch):
    size, ic, oc, k = 24, 20, 40, 3
    rng = np.random.default_rng(17)
    d = T.conv_desc(size, size, ic, k, k, oc, pad_same=True)
    x = rng.standard_normal((batch, ic * size * size)).astype(np.float32)
    w, b = rng.uniform(-0.2, 0.2, oc * ic * k * k).astype(np.float32), rng.standard_normal(oc).astype(np.float32)
    xd, y = T.to_device(x), T.DevBuf((batch, oc * size * size))
    T.conv2d_fwd(d, batch, xd, T.to_device(w), T.to_device(b), y)
    for flags in (0, T.NET_GRAPH):
        net = T.Net(W.build_layers(T, [("conv", size, size, ic, k, oc, True)]), batch, flags)
        net.set_param(0, 0, w)
        net.set_param(0, 1, b)
        net.forward(batch, xd)
        assert np.array_equal(y.numpy(), net.layer_out(0, batch))
        net.close()
