"""Infinities, NaN and values near the ends of fp32 in the convolution and fully-connected products: every sum that such
an operand is no part of stays what it is, and every other one is what fp32 gives. The reference is float64 with the
zeros around an image multiplied like any other value (0 times infinity is NaN), as the kernels do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FLT_MAX = float(np.finfo(np.float32).max)


def check(got, want, what):
    got, want = got.ravel().astype(np.float64), want.ravel()
    with np.errstate(invalid="ignore"):
        want = np.where(np.abs(want) > FLT_MAX, np.sign(want) * np.inf, want)
    assert np.array_equal(np.isnan(got), np.isnan(want)), (what, "NaN", np.isnan(got).sum(), np.isnan(want).sum())
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), (what, "infinities")
    rest = np.isfinite(want)
    ordinary = np.median(np.abs(want[rest]))
    # (sums of at most 2e4 products of the ordinary values, rounded after each; one large product beside them)
    got, want = got[rest], want[rest]
    assert (np.abs(got - want) <= 1e-4 * ordinary + 1e-6 * np.abs(want)).all(), what


def plant(a, rng, rows):
    """Exceptional values in as many rows of a (the largest one times an ordinary value does not overflow)."""
    flat = a.reshape(-1, a.shape[-1])
    for row, v in zip(rng.choice(len(flat), rows, replace=False), [np.inf, -np.inf, np.nan, 3e37, -2.5e32, 1e-41]):
        flat[row, rng.integers(a.shape[-1])] = v


def conv64(x, w, b, dy, ph, pw):
    """y, dx, dw, db in float64."""
    bs, ic, ih, iw = x.shape
    oc, _, r, s = w.shape
    oh, ow = dy.shape[2:]
    x, w, dy = (a.astype(np.float64) for a in (x, w, dy))
    xp = np.zeros((bs, ic, ih + 2 * ph, iw + 2 * pw)); xp[:, :, ph:ph + ih, pw:pw + iw] = x
    dyp = np.zeros((bs, oc, oh + 2 * (r - 1), ow + 2 * (s - 1))); dyp[:, :, r - 1:r - 1 + oh, s - 1:s - 1 + ow] = dy
    y, dxp, dw = np.zeros(dy.shape), np.zeros(xp.shape), np.zeros(w.shape)
    with np.errstate(invalid="ignore", over="ignore"):
        for fy in range(r):
            for fx in range(s):
                part = xp[:, :, fy:fy + oh, fx:fx + ow].reshape(bs, ic, -1)
                y += np.matmul(w[:, :, fy, fx], part).reshape(y.shape)
                dw[:, :, fy, fx] = sum(np.matmul(dy[i].reshape(oc, -1), part[i].T) for i in range(bs))
                at = dyp[:, :, r - 1 - fy:r - 1 - fy + xp.shape[2], s - 1 - fx:s - 1 - fx + xp.shape[3]].reshape(bs, oc, -1)
                dxp += np.matmul(w[:, :, fy, fx].T, at).reshape(dxp.shape)
        y += b.astype(np.float64).reshape(1, -1, 1, 1)
        db = dy.sum(axis=(0, 2, 3))
    return y, dxp[:, :, ph:ph + ih, pw:pw + iw], dw, db


THREE_PART = [
    # in_w, in_h, in_c, k, out_c, same, batch
    (64, 12, 16, 3, 64, True, 86),      # tiles of 64 columns, one chunk of channels
    (66, 17, 33, 3, 65, True, 26),      # scalar loads, channels past a chunk and a tile
    (30, 30, 64, 3, 40, False, 70),     # no padding
    (15, 33, 48, 3, 96, True, 90),      # tiles of 16 columns
    (53, 50, 20, 5, 40, True, 20),      # 5x5: dW in groups of filter rows
    (40, 40, 50, 1, 70, True, 26),      # 1x1
    (16, 16, 32, 5, 32, True, 21),      # dX shared by filter taps, in the launch with dW
    (8, 8, 32, 5, 64, True, 37),
]


FEW_TILES = [
    (12, 12, 5, 5, 9, True, 1),         # 225 and 125 indices: a last block of one and of thirteen
    (9, 7, 3, 3, 16, False, 1),         # 35 output pixels
    (10, 9, 24, 3, 8, True, 3),
]


@pytest.mark.parametrize("where", ["x", "w", "dy"])
@pytest.mark.parametrize("cfg", THREE_PART + FEW_TILES)
def test_convolution(T, cfg, where):
    iw, ih, ic, k, oc, same, bs = cfg
    rng = np.random.default_rng(31)
    d = T.conv_desc(iw, ih, ic, k, k, oc, pad_same=same)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic, ih, iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, (oc, ic, k, k)).astype(np.float32)
    dy = rng.standard_normal((bs, oc, oh, ow)).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    plant({"x": x, "w": w, "dy": dy}[where], rng, 6)
    out = [T.DevBuf((n,)) for n in (dy.size, x.size, w.size, oc)]
    xd, wd, dyd = (T.to_device(a.ravel()) for a in (x, w, dy))
    T.profile_begin()
    T.conv2d_fwd(d, bs, xd, wd, T.to_device(b), out[0])
    T.conv2d_bwd(d, bs, xd, wd, dyd, *out[1:])
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert tags & {"conv_bwd_pair", "conv_bwd_direct"} or cfg in THREE_PART and {"conv_fwd_x3", "conv_dx_x3"} <= tags, tags
    want = conv64(x, w, b, dy, *((k // 2, k // 2) if same else (0, 0)))
    for g, r, name in zip(out, want, ("y", "dx", "dw", "db")):
        check(g.numpy(), r, f"{cfg} {name}")


def test_ends_of_short_reductions(T):
    """The kernels for a few tiles fill the last block of 16 indices with the first weight and the last pixel, times
    zero: an infinity there reaches the sums that it is a part of, as an infinity."""
    iw, ih, ic, k, oc, bs = 9, 7, 5, 3, 9, 1
    rng = np.random.default_rng(34)
    d = T.conv_desc(iw, ih, ic, k, k, oc, pad_same=True)
    x = rng.uniform(0.5, 1, (bs, ic, ih, iw)).astype(np.float32)
    w = rng.uniform(0.5, 1, (oc, ic, k, k)).astype(np.float32)
    dy = rng.uniform(0.5, 1, (bs, oc, ih, iw)).astype(np.float32)
    b = np.zeros(oc, np.float32)
    w[0, 0, 0, 0] = x[-1, 2, -1, -1] = np.inf
    out = [T.DevBuf((n,)) for n in (dy.size, x.size, w.size, oc)]
    xd, wd, dyd = (T.to_device(a.ravel()) for a in (x, w, dy))
    T.conv2d_fwd(d, bs, xd, wd, T.to_device(b), out[0])
    T.conv2d_bwd(d, bs, xd, wd, dyd, *out[1:])
    for g, r, name in zip(out, conv64(x, w, b, dy, 1, 1), ("y", "dx", "dw", "db")):
        check(g.numpy(), r, name)


@pytest.mark.parametrize("where", ["x", "w"])
@pytest.mark.parametrize("dims", [(1028, 1012, 520), (8192, 2048, 64), (4096, 64, 2048)])
def test_fully_connected(T, W, dims, where):
    """Inference, and dX as an operator (x stands for dy there, w as it is)."""
    ni, no, bs = dims
    rng = np.random.default_rng(32)
    x = rng.standard_normal((bs, ni)).astype(np.float32)
    dy = rng.standard_normal((bs, no)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, (ni, no)).astype(np.float32)
    for a in (x, dy) if where == "x" else (w,):
        plant(a, rng, 6)
    net = T.Net(W.build_layers(T, [("fc", ni, no)]), bs, 0)
    net.set_param(0, 0, w)
    net.set_param(0, 1, np.zeros(no, np.float32))
    xd, dx = T.to_device(x), T.DevBuf(x.shape)
    T.profile_begin()
    net.forward(bs, xd)
    T.fc_bwd(ni, no, True, bs, xd, T.to_device(w.ravel()), T.to_device(dy), dx, None, None)
    assert {"fc_fwd_x3", "fc_dx_x3"} <= {e["tag"].split()[0] for e in T.profile_end()}
    with np.errstate(invalid="ignore", over="ignore"):
        check(net.layer_out(0, bs), x.astype(np.float64) @ w.astype(np.float64), f"{dims} y")
        check(dx.numpy(), dy.astype(np.float64) @ w.astype(np.float64).T, f"{dims} dx")
    net.close()


def test_packed_filters_behind_a_connection_table(T, W):
    """A net's inference reads packed filters; sums that are computed again read the weights and the table."""
    rng = np.random.default_rng(33)
    ic, oc, size, bs = 32, 48, 16, 300
    tbl = rng.integers(0, 2, ic * oc).astype(np.uint8)
    net = T.Net([T.L_conv(size, size, ic, 3, oc, True, tbl=tbl)], bs, T.NET_GRAPH)
    w = rng.uniform(-0.3, 0.3, (oc, ic, 3, 3)).astype(np.float32)
    on = tbl.reshape(ic, oc).T.astype(bool)
    w[~on, 0, 0] = np.inf                      # (never read)
    w[tuple(np.argwhere(on)[0])][1, 1] = 3e37   # (above 2^104, and no product of it overflows)
    b = rng.standard_normal(oc).astype(np.float32)
    net.set_param(0, 0, w.ravel())
    net.set_param(0, 1, b)
    x = rng.standard_normal((bs, ic, size, size)).astype(np.float32)
    plant(x, rng, 4)
    T.profile_begin()
    net.forward(bs, T.to_device(x.reshape(bs, -1)))
    assert any(e["tag"].startswith("conv_fwd_x3") for e in T.profile_end())
    w[~on] = 0
    dy = np.zeros((bs, oc, size, size), np.float32)
    check(net.layer_out(0, bs), conv64(x, w, b, dy, 1, 1)[0], "y")
    net.close()
