"""Forward convolution, dX and dW by the kernels that take any window, stride and size: against float64 where its tiles, chunks of
channels and phases end, and with infinities, NaN and the largest floats among the operands."""
import numpy as np
import pytest

from conftest import assert_close
from test_gpu_exceptional_values import check, plant

pytestmark = pytest.mark.gpu


def reference(x, w, b, dy, same, stride, dilation=(1, 1)):
    """y and dx in float64, a tap at a time. What lies outside the image, or outside the output, is a zero that is multiplied like
    any other value; padding::same puts k // 2 zeros in front."""
    x, w, dy = (a.astype(np.float64) for a in (x, w, dy))
    (ih, iw), (oh, ow), (kh, kw) = x.shape[2:], dy.shape[2:], w.shape[2:]
    (sh, sw), (eh, ew), (ph, pw) = stride, dilation, [k // 2 if same else 0 for k in (kh, kw)]

    def gather(a, rows, cols):
        inside = (rows >= 0) & (rows < a.shape[2]), (cols >= 0) & (cols < a.shape[3])
        g = np.zeros(a.shape[:2] + (len(rows), len(cols)))
        g[:, :, np.flatnonzero(inside[0])[:, None], np.flatnonzero(inside[1])] = a[:, :, rows[inside[0]][:, None], cols[inside[1]]]
        return g.reshape(a.shape[:2] + (-1,))

    y, dx = np.zeros(dy.shape), np.zeros(x.shape)
    with np.errstate(invalid="ignore", over="ignore"):
        for ky in range(kh):
            for kx in range(kw):
                y += np.matmul(w[:, :, ky, kx], gather(x, np.arange(oh) * sh + ky * eh - ph, np.arange(ow) * sw + kx * ew - pw)).reshape(y.shape)
                iy, ix = (np.flatnonzero((np.arange(n) + p - k) % s == 0) for n, p, k, s in ((ih, ph, ky, sh), (iw, pw, kx, sw)))
                part = np.matmul(w[:, :, ky, kx].T, gather(dy, (iy + ph - ky) // sh, (ix + pw - kx) // sw))
                dx[:, :, iy[:, None], ix] += part.reshape(dx.shape[:2] + (len(iy), len(ix)))
        return y + b.astype(np.float64).reshape(1, -1, 1, 1), dx


def within_fp32_sum(got, want, size):
    """A sum in fp32, each addition rounding to 2^-24 of a partial sum that grows as a random walk, is 0.64 * 2^-24 of
    the sum of absolute products (size) away, rms; no element is twelve times as far."""
    return (np.abs(got.ravel() - want.ravel()) <= 8 * 2.0 ** -24 * size.ravel()).all()


CASES = [
    # in_w, in_h, in_c, kw, kh, out_c, same, (sh, sw), batch; the directions that take the kernel
    (45, 37, 21, 5, 5, 45, False, (2, 2), 19, "fb"),   # 9, 6, 6 and 4 taps a phase, a last group of 5 channels
    (31, 91, 3, 7, 7, 20, True, (2, 2), 40, "fb"),     # three channels: reductions of one group
    (17, 15, 79, 7, 7, 4, True, (1, 1), 60, "fb"),     # tiles of several images, several chunks
    (26, 32, 9, 3, 3, 69, True, (1, 1), 40, "b"),      # dX of 9 channels
    (34, 21, 58, 5, 5, 3, False, (1, 1), 92, "f"),     # 3 of 16 rows in use
    (50, 47, 40, 3, 2, 130, True, (3, 1), 24, "fb"),   # unequal strides and window sides, channels past two workgroups
    (21, 20, 70, 3, 3, 65, True, (2, 1), 33, "fb"),
    (96, 5, 33, 1, 7, 40, True, (2, 2), 60, "b"),      # one column of taps: phases without a tap
    (65, 40, 26, 5, 5, 30, True, (1, 1), 12, "b"),     # in the place of the stride-1 kernel
    (9, 9, 64, 3, 3, 64, False, (2, 2), 300, "fb"),    # images of 16 outputs
]


def operands(T, cfg, rng):
    iw, ih, ic, kw, kh, oc, same, (sh, sw), bs = cfg[:9]
    d = T.conv_desc(iw, ih, ic, kw, kh, oc, pad_same=same, w_stride=sw, h_stride=sh)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic, ih, iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, (oc, ic, kh, kw)).astype(np.float32)
    return d, x, w, rng.standard_normal(oc).astype(np.float32), rng.standard_normal((bs, oc, oh, ow)).astype(np.float32)


def run(T, d, x, w, b, dy):
    y, dx = T.to_device(np.full(dy.size, 7, np.float32)), T.to_device(np.full(x.size, 7, np.float32))
    xd, wd, bd, dyd = (T.to_device(a.ravel()) for a in (x, w, b, dy))
    T.profile_begin()
    T.conv2d_fwd(d, len(x), xd, wd, bd, y)
    T.conv2d_bwd(d, len(x), xd, wd, dyd, dx, None, None)
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    return y.numpy(), dx.numpy(), "".join(k for k, t in (("f", "conv_fwd_any_x3"), ("b", "conv_dx_any_x3")) if t in tags)


@pytest.mark.parametrize("cfg", CASES)
def test_against_float64(T, cfg):
    d, x, w, b, dy = operands(T, cfg, np.random.default_rng(41))
    y, dx, taken = run(T, d, x, w, b, dy)
    assert taken == cfg[9]
    sizes = reference(*(np.abs(a) for a in (x, w, b, dy)), cfg[6], cfg[7])
    for got, want, size, name in zip((y, dx), reference(x, w, b, dy, cfg[6], cfg[7]), sizes, ("y", "dx")):
        assert_close(got, want.ravel(), what=f"{cfg} {name}")
        assert within_fp32_sum(got, want, size), name
        # No further from float64 than a sum in fp32: K terms in order, each addition rounding to 2^-24 of a partial sum
        # that grows as a random walk, leave 2^-24 sqrt(K / 6) of the result; six bits under that and 2^-23 of the parts.
        k = cfg[3] * cfg[4] * cfg[2 if name == "y" else 5] / (1 if name == "y" else cfg[7][0] * cfg[7][1])
        assert np.linalg.norm(got - want.ravel()) <= 2 ** -24 * (2 + np.sqrt(k / 6)) * np.linalg.norm(want)


def test_dilation(T):
    iw, ih, ic, k, oc, bs = 40, 33, 20, 3, 40, 30
    rng = np.random.default_rng(42)
    d = T.conv_desc(iw, ih, ic, k, k, oc, pad_same=False, w_stride=2, h_stride=1, w_dilation=3, h_dilation=2)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((bs, ic, ih, iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, (oc, ic, k, k)).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    y = T.DevBuf((bs * oc * oh * ow,))
    T.profile_begin()
    T.conv2d_fwd(d, bs, T.to_device(x.ravel()), T.to_device(w.ravel()), T.to_device(b), y)
    assert any(e["tag"].startswith("conv_fwd_any_x3") for e in T.profile_end())
    want = reference(x, w, b, np.zeros((bs, oc, oh, ow), np.float32), False, (1, 2), (2, 3))[0]
    assert_close(y.numpy(), want.ravel(), what="y")


@pytest.mark.parametrize("where", ["x", "w", "dy"])
@pytest.mark.parametrize("cfg", [CASES[0], CASES[9]])
def test_exceptional_values(T, cfg, where):
    rng = np.random.default_rng(43)
    d, x, w, b, dy = operands(T, cfg, rng)
    plant({"x": x, "w": w, "dy": dy}[where], rng, 6)
    y, dx, taken = run(T, d, x, w, b, dy)
    assert taken == "fb"
    for got, want, name in zip((y, dx), reference(x, w, b, dy, cfg[6], cfg[7]), ("y", "dx")):
        check(got, want, f"{cfg} {name}")


DW_CASES = [
    # as above, and what the launch is called with gradients stored and added (a train step keeps db apart)
    (45, 37, 21, 5, 5, 45, False, (2, 2), 19, "conv_dw_db_any", "conv_dw_any"),
    (59, 30, 46, 5, 5, 3, False, (1, 1), 40, "conv_dw_db_any", "conv_dw_any"),     # channels shared by two tiles of columns
    (31, 91, 3, 7, 7, 20, True, (2, 2), 260, "conv_dw_db_any", "conv_dw_any"),     # one or two channels a tile
    (23, 19, 33, 7, 3, 70, True, (3, 1), 60, "conv_dw_db_any", "conv_dw_any"),     # two workgroups of output channels
    (12, 11, 85, 1, 7, 3, True, (2, 2), 600, "conv_dw_db_any", "conv_dw_any"),     # several images a chunk
    (12, 11, 85, 5, 5, 3, True, (1, 1), 200, "conv_dw_db_any", "conv_dw_any"),
    (22, 20, 32, 3, 3, 3, False, (2, 2), 900, "conv_dw_any", "conv_dw_any"),       # 288 columns: db is no part of the tiles
]


def weight_gradient(x, dy, kh, kw, same, stride):
    x, dy = x.astype(np.float64), dy.astype(np.float64)
    (oh, ow), (sh, sw), (ph, pw) = dy.shape[2:], stride, [k // 2 if same else 0 for k in (kh, kw)]
    xp = np.zeros(x.shape[:2] + (x.shape[2] + 2 * kh + sh, x.shape[3] + 2 * kw + sw))
    xp[:, :, ph:ph + x.shape[2], pw:pw + x.shape[3]] = x
    dw = np.zeros((dy.shape[1], x.shape[1], kh, kw))
    flat = dy.transpose(1, 0, 2, 3).reshape(dy.shape[1], -1)
    with np.errstate(invalid="ignore", over="ignore"):
        for ky in range(kh):
            for kx in range(kw):
                part = xp[:, :, ky:ky + (oh - 1) * sh + 1:sh, kx:kx + (ow - 1) * sw + 1:sw]
                dw[:, :, ky, kx] = np.matmul(flat, part.transpose(0, 2, 3, 1).reshape(-1, x.shape[1]))
        return dw, dy.sum(axis=(0, 2, 3))


@pytest.mark.parametrize("accumulate", [0, 1])
@pytest.mark.parametrize("cfg", DW_CASES)
def test_weight_gradient_against_float64(T, cfg, accumulate):
    rng = np.random.default_rng(44)
    d, x, w, b, dy = operands(T, cfg, rng)
    before = rng.standard_normal(w.size + b.size).astype(np.float32)
    dw, db = T.to_device(before[:w.size].copy()), T.to_device(before[w.size:].copy())
    T.profile_begin()
    T.conv2d_bwd(d, len(x), T.to_device(x.ravel()), T.to_device(w.ravel()), T.to_device(dy.ravel()), None, dw, db, accumulate)
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert cfg[9 + accumulate] in tags, tags
    want = weight_gradient(x, dy, cfg[4], cfg[3], cfg[6], cfg[7])
    sizes = weight_gradient(np.abs(x), np.abs(dy), cfg[4], cfg[3], cfg[6], cfg[7])
    for got, ref, size, old, name in zip((dw.numpy(), db.numpy()), want, sizes, (before[:w.size], before[w.size:]), ("dw", "db")):
        ref = ref.ravel() + (old if accumulate else 0)
        assert within_fp32_sum(got, ref, size.ravel() + (np.abs(old) if accumulate else 0)), name
        assert_close(got, ref, what=f"{cfg} {name}")
        # K products in order in at least 64 slices: the bound of the sums above for K / 64 terms and for 64
        k = dy.size / dy.shape[1]
        assert np.linalg.norm(got - ref) <= 2 ** -24 * (3 + np.sqrt(k / 64 / 6) + np.sqrt(64 / 6)) * np.linalg.norm(ref)


@pytest.mark.parametrize("where", ["x", "dy"])
def test_weight_gradient_of_exceptional_values(T, where):
    cfg = (59, 30, 46, 5, 5, 3, False, (1, 1), 13)   # (18590 pixels: a last piece of 14)
    rng = np.random.default_rng(45)
    d, x, w, b, dy = operands(T, cfg, rng)
    plant({"x": x, "dy": dy}[where], rng, 6)
    (x if where == "x" else dy)[-1, 2, -1, -1] = np.inf
    dw, db = T.DevBuf((w.size,)), T.DevBuf((b.size,))
    T.profile_begin()
    T.conv2d_bwd(d, len(x), T.to_device(x.ravel()), T.to_device(w.ravel()), T.to_device(dy.ravel()), None, dw, db)
    assert any(e["tag"].startswith("conv_dw_db_any") for e in T.profile_end())
    for got, ref, name in zip((dw.numpy(), db.numpy()), weight_gradient(x, dy, 5, 5, False, (1, 1)), ("dw", "db")):
        check(got, ref, name)


@pytest.mark.parametrize("cfg", [
    # (us of the forward product by the generic kernel / by the one of any size)
    (94, 10, 92, 1, 1, 11, True, (1, 1), 54, False),    # 14 / 28
    (70, 59, 65, 1, 5, 56, False, (2, 2), 23, False),   # 33 / 53
    (29, 82, 86, 3, 1, 2, False, (2, 2), 59, False),    # 26 / 39
    (44, 43, 2, 7, 7, 39, True, (2, 2), 72, False),     # 17 / 24
    (41, 70, 74, 7, 7, 6, True, (2, 2), 120, True),     # 717 / 311
    (19, 74, 31, 7, 5, 2, True, (1, 1), 97, True),      # 211 / 73
])
def test_forward_product_takes_the_faster_kernel(T, cfg):
    d, x, w, b, dy = operands(T, cfg, np.random.default_rng(46))
    assert ("f" in run(T, d, x, w, b, dy)[2]) == cfg[9]


@pytest.mark.parametrize("cfg", [
    # (us of dX by the stride-1 kernel / by the one of any size)
    (59, 13, 51, 5, 5, 139, True, (1, 1), 2, False),   # 22 / 56
    (55, 7, 23, 3, 3, 157, True, (1, 1), 8, False),    # 16 / 31
    (77, 9, 94, 5, 5, 113, False, (1, 1), 2, False),   # 30 / 51
    (43, 31, 94, 3, 3, 74, True, (1, 1), 6, True),     # 40 / 25
    (19, 89, 64, 3, 3, 21, True, (1, 1), 11, True),    # 26 / 16
    # (... by the vector kernel of a first layer)
    (70, 25, 3, 4, 4, 127, True, (1, 1), 83, False),   # 104 / 160
    (29, 61, 2, 7, 5, 110, True, (1, 1), 76, False),   # 164 / 261
    (41, 40, 3, 7, 7, 105, True, (1, 1), 101, True),   # 379 / 219
    (18, 15, 1, 7, 7, 116, True, (1, 1), 1, True),     # 155 / 29
])
def test_input_gradient_takes_the_faster_kernel(T, cfg):
    d, x, w, b, dy = operands(T, cfg, np.random.default_rng(47))
    assert ("b" in run(T, d, x, w, b, dy)[2]) == cfg[9]


@pytest.mark.parametrize("cfg", [
    # (us of dW and db by the generic kernel / by the one of any size)
    (52, 71, 24, 3, 3, 114, True, (2, 2), 47, False),   # 56 / 97, 68 with whole rounds in the choice of its tile
    (65, 19, 123, 3, 5, 109, True, (1, 1), 21, False),  # 157 / 222, 176
    (59, 56, 46, 5, 5, 3, True, (1, 1), 69, True),      # 286 / 141
    (48, 85, 55, 7, 7, 12, True, (1, 1), 26, True),     # 362 / 155
])
def test_weight_gradient_takes_the_faster_kernel(T, cfg):
    d, x, w, b, dy = operands(T, cfg, np.random.default_rng(48))
    dw, db = T.DevBuf((w.size,)), T.DevBuf((b.size,))
    T.profile_begin()
    T.conv2d_bwd(d, len(x), T.to_device(x.ravel()), T.to_device(w.ravel()), T.to_device(dy.ravel()), None, dw, db)
    assert any(e["tag"].startswith("conv_dw_db_any") for e in T.profile_end()) == cfg[9]


NET = dict(w=45, h=37, ci=3, mid=21, co=45, k=5, batch=19)   # 3x3 to 21 channels, then 5x5 at stride 2 to 45: ragged everywhere


def tags_of(T, f):
    T.profile_begin()
    f()
    return {e["tag"].split()[0] for e in T.profile_end()}


@pytest.mark.parametrize("exceptional", [False, True])
@pytest.mark.parametrize("kind", ["relu", "tanh", "sigmoid"])
def test_inference_writes_the_activation_behind_it(T, kind, exceptional):
    """A net's forward pass takes the pointwise activation along: the bits of the two operators, and float64."""
    n, rng = NET, np.random.default_rng(51)
    d, x, w, b, dy = operands(T, (n["w"], n["h"], n["mid"], n["k"], n["k"], n["co"], False, (2, 2), n["batch"]), rng)
    if exceptional:
        plant(x, rng, 6)
    net = T.Net([T.L_conv(n["w"], n["h"], n["mid"], n["k"], n["co"], stride=2), T.L_act(kind)], n["batch"], T.NET_FUSE_ACT_GRAD)
    net.set_param(0, 0, w.ravel())
    net.set_param(0, 1, b)
    xd, y, a = T.to_device(x), T.DevBuf((dy.size,)), T.DevBuf((dy.size,))
    tags = tags_of(T, lambda: net.forward(n["batch"], xd))
    assert "conv_fwd_any_x3" in tags and not any(t.startswith("act") for t in tags), tags
    T.conv2d_fwd(d, n["batch"], xd, T.to_device(w.ravel()), T.to_device(b), y)
    T.act_fwd(kind, n["batch"], dy.size // n["batch"], y, a)
    assert np.array_equal(net.layer_out(0, n["batch"]).ravel(), y.numpy(), equal_nan=True)
    assert np.array_equal(net.layer_out(1, n["batch"]).ravel(), a.numpy(), equal_nan=True)
    check(y.numpy(), reference(x, w, b, dy, False, (2, 2))[0], kind)
    net.close()


@pytest.mark.parametrize("exceptional", [False, True])
@pytest.mark.parametrize("kind", ["relu", "tanh", "sigmoid"])
def test_input_gradient_folds_the_activation_in_front(T, kind, exceptional):
    """A train step's dX through the activation between two convolutions, against float64 on the step's own outputs."""
    n, rng = NET, np.random.default_rng(52)
    _, x, w0, b0, _ = operands(T, (n["w"], n["h"], n["ci"], 3, 3, n["mid"], True, (1, 1), n["batch"]), rng)
    _, _, w1, b1, dy = operands(T, (n["w"], n["h"], n["mid"], n["k"], n["k"], n["co"], False, (2, 2), n["batch"]), rng)
    layers = [T.L_conv(n["w"], n["h"], n["ci"], 3, n["mid"], pad_same=True), T.L_act(kind),
              T.L_conv(n["w"], n["h"], n["mid"], n["k"], n["co"], stride=2)]
    net = T.Net(layers, n["batch"], T.NET_FUSE_ACT_GRAD)
    for i, w, b in ((0, w0, b0), (2, w1, b1)):
        net.set_param(i, 0, w.ravel())
        net.set_param(i, 1, b)
    t = rng.standard_normal(dy.shape).astype(np.float32)
    if exceptional:
        plant(t, rng, 4)   # (infinities and NaN of dY: sums that are computed again, then multiplied by the activation's gradient)
    tags = tags_of(T, lambda: net.train_step(None, "mse", n["batch"], T.to_device(x), T.to_device(t), do_update=False))
    assert "conv_dx_any_x3" in tags and not any(g.startswith("act_bwd") for g in tags), tags
    a, y = net.layer_out(1, n["batch"]).reshape(n["batch"], n["mid"], n["h"], n["w"]), net.layer_out(2, n["batch"]).reshape(dy.shape)
    dy = ((y - t) * np.float32(2.0 / (dy.size // n["batch"]))).astype(np.float32)
    a64 = a.astype(np.float64)
    factor = {"relu": (a64 > 0) * 1.0, "tanh": 1 - a64 * a64, "sigmoid": a64 * (1 - a64)}[kind]
    with np.errstate(invalid="ignore"):
        want = reference(a, w1, b1, dy, False, (2, 2))[1] * factor
    got = net.layer_dx(1, n["batch"]).ravel()
    if exceptional:
        assert not np.isfinite(got).all()
        on = factor.ravel() != 0   # (behind a rectifier that is off: 0, or NaN where the sum is not finite)
        check(got[on], want.ravel()[on], kind)
        assert np.array_equal(got[~on], want.ravel()[~on], equal_nan=True)
    else:
        assert_close(got, want.ravel(), what=kind)
        k = n["k"] ** 2 * n["co"] / 4
        assert np.linalg.norm(got - want.ravel()) <= 2 ** -24 * (6 + np.sqrt(k / 6)) * np.linalg.norm(want)
    net.close()
