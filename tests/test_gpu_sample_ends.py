"""The small net's step where it begins with a convolution, activations and pools, and a second convolution: the front
and the back of its chain run a channel a workgroup while there is a compute unit for each. Every tensor against the
oracle, at the ends of those kernels' tiles and on both sides of the line between the two forms."""
import numpy as np
import pytest

from conftest import assert_close
from test_gpu_sample_step import FUSE, SAMPLE, build

pytestmark = pytest.mark.gpu

TABLE = [[(2 * ci + co) % 3 != 0 for co in range(9)] for ci in range(5)]
NETS = {
    # a first plane of more pixels than threads; rows of the second one that are no multiple of four, in two chunks of units
    "wide": ([("conv", 40, 38, 1, 3, 4, True), ("act", "tanh"), ("maxpool", 40, 38, 4, 2), ("act", "sigmoid"),
              ("conv", 20, 19, 4, 5, 8, True), ("act", "tanh"), ("maxpool", 20, 19, 8, 3),
              ("fc", 8 * 6 * 6, 5)], "mse", "sgd"),
    # five layers in front (one more than travel ahead), table behind, windows clipped by the edge
    "deep_front": ([("conv", 17, 15, 3, 5, 5, True), ("act", "tanh"), ("act", "sigmoid"), ("maxpool", 17, 15, 5, 2),
                    ("act", "tanh"), ("act", "leaky_relu", (0.2, 0.0)), ("conv", 8, 7, 5, 3, 9, False, TABLE),
                    ("act", "tanh"), ("fc", 9 * 6 * 5, 4), ("act", "softmax")], "ce_multiclass", "momentum"),
    # 64 output channels are the most that the back kernel sums over; 65 stay in one launch
    "k64": ([("conv", 9, 9, 2, 3, 3, False), ("conv", 7, 7, 3, 3, 64, True), ("act", "tanh"), ("fc", 64 * 49, 3)], "mse", "adagrad"),
    "k65": ([("conv", 9, 9, 2, 3, 3, False), ("conv", 7, 7, 3, 3, 65, True), ("act", "tanh"), ("fc", 65 * 49, 3)], "mse", "adagrad"),
    # an average pool of odd height behind it, two channels
    "two": ([("conv", 12, 10, 1, 5, 2, False), ("act", "sigmoid"), ("avepool", 8, 6, 2, 2), ("conv", 4, 3, 2, 3, 4, True),
             ("fc", 48, 6), ("act", "sigmoid")], "ce", "adam"),
}
ENDS = {"wide": 64, "deep_front": 51, "k64": 85, "k65": None, "two": 128}   # the largest batch of the split form


@pytest.mark.parametrize("name", list(NETS))
@pytest.mark.parametrize("batch", [1, 3, "last", "past"])
def test_every_tensor_matches_oracle(T, O, W, name, batch):
    split = ENDS[name] is not None
    if not isinstance(batch, int):
        if not split:
            pytest.skip("this net has one form")
        split, batch = batch == "last", ENDS[name] + (batch == "past")
    spec, params, x, t, batch, loss, kind, _, net, ref = build(T, O, W, name, batch, SAMPLE | FUSE, nets=NETS)
    xd, td = T.to_device(x), T.to_device(t)
    T.profile_begin()
    net.train_step(None, loss, batch, xd, td, do_update=False)
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert ("tiny_net_front" in tags) == ("tiny_net_back" in tags) == split, tags
    ref.train_step(O.opt_desc(kind), loss, x, t, do_update=False)
    for i, l in enumerate(spec):
        assert_close(net.layer_out(i, batch), ref.layer_out(i, batch), what=f"layer {i} output")
        assert_close(net.layer_dx(i, batch), ref.layer_dx(i, batch), what=f"layer {i} dX")
        if l[0] == "maxpool":
            assert np.array_equal(net.layer_argmax(i, batch).astype(np.int64), ref.layer_argmax(i, batch))
        if net.param_size(i, 0):
            assert_close(net.layer_grad(i, 0), ref.layer_dw(i), what=f"layer {i} dW")
            assert_close(net.layer_grad(i, 1), ref.layer_db(i), what=f"layer {i} db")
    net.close()


# nets whose parameter gradients take every road: channel pairs of 3x3 and 5x5 windows, of any window and stride, outer
# products in words and one by one, average pools, tables
PARAM_NETS = {
    "wide": NETS["wide"], "deep_front": NETS["deep_front"], "two": NETS["two"],
    "any_window": ([("conv", 14, 13, 2, 4, 5, False), ("act", "tanh"), ("avepool", 11, 10, 5, 1), ("conv", 11, 10, 5, 2, 6, False),
                    ("act", "sigmoid"), ("fc", 6 * 90, 7)], "mse", "adam"),
    "fc": ([("fc", 37, 24), ("act", "tanh"), ("fc", 24, 36), ("act", "sigmoid"), ("fc", 36, 5)], "mse", "adam"),
    # many channel pairs of small planes, a wave a pair: blocks of input channels that overlap, a table, one block of two channels
    "many_pairs": ([("conv", 9, 8, 3, 3, 11, True), ("act", "tanh"), ("conv", 9, 8, 11, 3, 40, True,
                    [[(ci + 2 * co) % 3 != 0 for co in range(40)] for ci in range(11)]), ("act", "sigmoid"),
                    ("fc", 40 * 72, 4)], "mse", "adam"),
    "many_pairs_5x5": ([("conv", 9, 8, 2, 5, 120, False), ("act", "tanh"), ("fc", 120 * 20, 3)], "mse", "adam"),
    "matvec": ([("conv", 5, 5, 3, 5, 8, False, [[(ci + co) % 2 == 0 for co in range(8)] for ci in range(3)]), ("act", "tanh"),
                ("fc", 8, 3)], "mse", "adam"),
}


@pytest.mark.parametrize("kind", ["sgd", "momentum", "adam", "adagrad", "rmsprop", "adamax", "nesterov"])
@pytest.mark.parametrize("name,batch", [("wide", 16), ("deep_front", 32), ("deep_front", 33), ("two", 1), ("any_window", 31),
                                        ("any_window", 50), ("fc", 32), ("fc", 64), ("fc", 70), ("matvec", 17), ("matvec", 100)])
def test_gradients_and_updates_of_one_group_and_of_several(T, O, W, name, batch, kind):
    """Small batches are updated by the launch that adds up the gradients; larger ones leave slices. Gradients against the
    oracle; updates, of a step that adds to the gradients of a pass without one, against the layer-by-layer step."""
    spec, params, x, t, batch, loss, _, _, net, ref = build(T, O, W, name, batch, SAMPLE | FUSE, nets=PARAM_NETS)
    *_, replay, _ = build(T, O, W, name, batch, SAMPLE | FUSE | 2, nets=PARAM_NETS)
    *_, layered, _ = build(T, O, W, name, batch, FUSE, nets=PARAM_NETS)
    xd, td = T.to_device(x), T.to_device(t)
    alpha = {"sgd": 1e-3, "momentum": 1e-3, "nesterov": 1e-3}.get(kind, 1e-2)
    opts = [T.opt_desc(kind, alpha=alpha) for _ in range(3)]
    for m in (net, replay, layered):
        m.train_step(None, loss, batch, xd, td, do_update=False)
    ref.train_step(O.opt_desc(kind), loss, x, t, do_update=False)
    grads = {(i, w): (ref.layer_dw(i) if w == 0 else ref.layer_db(i)).copy() for i, w, _ in params}
    for (i, w), want in grads.items():
        assert_close(net.layer_grad(i, w), want, what=f"gradient {i}.{w}")
    for k, m in enumerate((net, replay, layered)):
        for _ in range(2):
            m.train_step(opts[k], loss, batch, xd, td)
    divides = kind in ("adam", "adagrad", "rmsprop", "adamax")
    for i, w, a in params:
        got, want = net.get_param(i, w), layered.get_param(i, w)
        assert np.array_equal(got, replay.get_param(i, w))
        if divides:
            # a gradient's relative error of 1e-4 (of its tensor's rms) moves a weight by up to alpha times itself over the
            # gradient's own size: elements below a hundredth of the rms are left out, the others get 1e-2 of a step
            g = np.abs(grads[(i, w)].ravel())
            on = g > 1e-2 * np.sqrt(np.mean(g * g))
            assert np.abs(got.ravel() - want.ravel())[on].max(initial=0.0) <= 2 * 2 * 1e-2 * alpha, f"{kind} parameter {i}.{w}"
        else:
            assert_close(got, want, what=f"{kind} parameter {i}.{w}")
        assert not net.layer_grad(i, w).any()
    assert opts[0].b1_t == opts[1].b1_t == opts[2].b1_t and opts[0].b2_t == opts[1].b2_t == opts[2].b2_t
    for m in (net, replay, layered):
        m.close()


def roads_of(T, step):
    T.profile_begin()
    step()
    return {e["tag"].split()[0] for e in T.profile_end()}


@pytest.mark.parametrize("name,batch,road", [("many_pairs", 65, "waves"), ("many_pairs", 200, "waves"), ("many_pairs", 12, None),
                                             ("many_pairs_5x5", 100, "waves"), ("any_window", 9, "any")])
def test_gradients_of_many_pairs_and_of_any_window(T, O, W, name, batch, road):
    spec, params, x, t, batch, loss, kind, _, net, ref = build(T, O, W, name, batch, SAMPLE | FUSE, nets=PARAM_NETS)
    xd, td = T.to_device(x), T.to_device(t)
    tags = roads_of(T, lambda: net.train_step(None, loss, batch, xd, td, do_update=False))
    assert "tiny_net_param_grads" + ("_" + road if road else "") in tags, tags
    ref.train_step(O.opt_desc(kind), loss, x, t, do_update=False)
    for i, w, _ in params:
        assert_close(net.layer_grad(i, w), ref.layer_dw(i) if w == 0 else ref.layer_db(i), what=f"gradient {i}.{w}")
    opt = T.opt_desc(kind, alpha=1e-3)
    tags = roads_of(T, lambda: net.train_step(opt, loss, batch, xd, td))
    assert any(tag.startswith("opt_") for tag in tags) == (batch > 12 or road == "any"), tags
    net.close()


# convolutions whose gradients are added up sample by sample: rows a multiple of eight words apart, in 32 lanes a weight; a first
# layer whose input gradient runs in the same launch, with a table and strides behind it; an average pool beside them
ROWS_NETS = {
    "rows32": ([("conv", 32, 32, 1, 4, 8, True), ("act", "tanh"), ("maxpool", 32, 32, 8, 2), ("fc", 2048, 10)], "mse", "sgd"),
    "first_dx": ([("conv", 16, 16, 2, 3, 5, True), ("act", "sigmoid"), ("avepool", 16, 16, 5, 2),
                  ("conv", 8, 8, 5, 1, 9, False, TABLE), ("act", "tanh"), ("fc", 9 * 64, 7)], "mse", "momentum"),
}


@pytest.mark.parametrize("name", list(ROWS_NETS))
@pytest.mark.parametrize("batch", [1, 2, 4, 8, 9, 70])
def test_sums_sample_by_sample(T, O, W, name, batch):
    """Gradients against the oracle; one step's update, of a few samples by the same launch, against the layer-by-layer step."""
    spec, params, x, t, batch, loss, kind, _, net, ref = build(T, O, W, name, batch, SAMPLE | FUSE, nets=ROWS_NETS)
    *_, layered, _ = build(T, O, W, name, batch, FUSE, nets=ROWS_NETS)
    xd, td = T.to_device(x), T.to_device(t)
    tags = roads_of(T, lambda: net.train_step(None, loss, batch, xd, td, do_update=False))
    assert "tiny_net_param_grads_any" in tags, tags
    ref.train_step(O.opt_desc(kind), loss, x, t, do_update=False)
    assert_close(net.layer_dx(0, batch), ref.layer_dx(0, batch), what="input gradient")
    for i, w, _ in params:
        assert_close(net.layer_grad(i, w), ref.layer_dw(i) if w == 0 else ref.layer_db(i), what=f"gradient {i}.{w}")
    layered.train_step(None, loss, batch, xd, td, do_update=False)
    tags = roads_of(T, lambda: net.train_step(T.opt_desc(kind, alpha=1e-3), loss, batch, xd, td))
    assert any(tag.startswith("opt_") for tag in tags) == (batch > {"rows32": 1, "first_dx": 2}[name]), tags
    layered.train_step(T.opt_desc(kind, alpha=1e-3), loss, batch, xd, td)
    for i, w, _ in params:
        assert_close(net.get_param(i, w), layered.get_param(i, w), what=f"parameter {i}.{w}")
    net.close()
    layered.close()


def test_sums_sample_by_sample_are_the_shorter_part(T, O, W):
    """Sixteen samples of the first of these nets: its gradients took 84 us where the chain takes 54, now 7."""
    spec, params, x, t, batch, loss, kind, _, net, _ = build(T, O, W, "rows32", 16, SAMPLE | FUSE, nets=ROWS_NETS)
    xd, td = T.to_device(x), T.to_device(t)
    opt = T.opt_desc(kind, alpha=1e-6)
    for _ in range(3):
        net.train_step(opt, loss, batch, xd, td)
    T.profile_begin()
    for _ in range(10):
        net.train_step(opt, loss, batch, xd, td)
    us = {e["tag"].split()[0]: e["avg_us"] for e in T.profile_end()}
    assert us["tiny_net_param_grads_any"] < 0.5 * us["tiny_net_step"], us
    net.close()


@pytest.mark.parametrize("batch", [1, 6, 40])
def test_strided_convolutions_match_oracle(T, O, batch):
    """Windows and strides that no fast form takes, one of them behind a 3x3 window of stride 1 (the first layer's dX and a
    channel pair's gradients beside them)."""
    def layers(L):
        return [L.L_conv(13, 12, 2, 3, 5, pad_same=True), L.L_act("tanh"), L.L_conv(13, 12, 5, 4, 6, stride=2), L.L_act("sigmoid"),
                L.L_conv(5, 5, 6, 3, 7, pad_same=True, stride=3, has_bias=False), L.L_act("tanh"), L.L_fc(7 * 4, 3)]

    rng = np.random.default_rng(5)
    net, ref = T.Net(layers(T), batch, SAMPLE | FUSE), O.OracleNet(layers(O), batch)
    for i, which, n in net.params():
        a = rng.uniform(-0.4, 0.4, n).astype(np.float32)
        net.set_param(i, which, a)
        (ref.weight(i) if which == 0 else ref.bias(i))[:] = a
    x = rng.standard_normal((batch, net.in_size())).astype(np.float32)
    t = rng.uniform(-0.8, 0.8, (batch, net.out_size())).astype(np.float32)
    tags = roads_of(T, lambda: net.train_step(None, "mse", batch, T.to_device(x), T.to_device(t), do_update=False))
    assert "tiny_net_param_grads_any" in tags, tags
    ref.train_step(O.opt_desc("sgd"), "mse", x, t, do_update=False)
    for i in range(net.n):
        assert_close(net.layer_out(i, batch), ref.layer_out(i, batch), what=f"layer {i} output")
        assert_close(net.layer_dx(i, batch), ref.layer_dx(i, batch), what=f"layer {i} dX")
    for i, w, _ in net.params():
        assert_close(net.layer_grad(i, w), ref.layer_dw(i) if w == 0 else ref.layer_db(i), what=f"gradient {i}.{w}")
    net.close()


@pytest.mark.parametrize("k,same,in_c,out_c", [(3, False, 2, 4), (3, True, 2, 4), (5, True, 1, 3), (5, False, 2, 3), (3, True, 9, 40)])
@pytest.mark.parametrize("batch", [3, 90])
def test_infinities_stay_out_of_sums_that_they_are_no_part_of(T, O, k, same, in_c, out_c, batch):
    """Minus infinity at corners of the input: relu makes a zero of what they reach, so that the first layer's weight gradient has a NaN
    (infinity times zero) exactly where one of them meets an output pixel, in the oracle's sums as well."""
    w, h = 10, 9
    ow, oh = (w, h) if same else (w - k + 1, h - k + 1)

    def layers(L):
        return [L.L_conv(w, h, in_c, k, out_c, pad_same=same), L.L_act("relu"), L.L_conv(ow, oh, out_c, 3, 5, pad_same=True),
                L.L_act("tanh"), L.L_fc(5 * ow * oh, 2)]

    rng = np.random.default_rng(8)
    net, ref = T.Net(layers(T), batch, SAMPLE | FUSE), O.OracleNet(layers(O), batch)
    for i, which, n in net.params():
        a = rng.uniform(0.05, 0.4, n).astype(np.float32) if i == 0 else rng.uniform(-0.3, 0.3, n).astype(np.float32)
        net.set_param(i, which, a)
        (ref.weight(i) if which == 0 else ref.bias(i))[:] = a
    x = rng.standard_normal((batch, in_c, h, w)).astype(np.float32)
    x[0, 0, 0, 0] = x[1, in_c - 1, h - 1, w - 1] = x[2, 0, 0, w - 1] = -np.inf
    x = x.reshape(batch, -1)
    t = rng.uniform(-0.8, 0.8, (batch, 2)).astype(np.float32)
    tags = roads_of(T, lambda: net.train_step(None, "mse", batch, T.to_device(x), T.to_device(t), do_update=False))
    assert {"tiny_net_step"} <= tags and any(tag.startswith("tiny_net_param_grads") for tag in tags), tags
    ref.train_step(O.opt_desc("sgd"), "mse", x, t, do_update=False)

    def same_values(got, want, what):
        got, want = np.asarray(got).ravel(), np.asarray(want).ravel()
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)), what
        on = np.isfinite(want)
        assert_close(got[on], want[on], what=what)

    for i in range(net.n):
        same_values(net.layer_out(i, batch), ref.layer_out(i, batch), f"layer {i} output")
        same_values(net.layer_dx(i, batch), ref.layer_dx(i, batch), f"layer {i} dX")
    for i, which, _ in net.params():
        same_values(net.layer_grad(i, which), ref.layer_dw(i) if which == 0 else ref.layer_db(i), f"gradient {i}.{which}")
    dw = ref.layer_dw(0)
    assert np.isnan(dw).any() and np.isfinite(dw).any()   # (the test's point)
    net.close()


HELD_NETS = {
    # 16 rows a thread are the most: 24 pieces of a row, 16 ranges of channels
    "k256": ([("conv", 8, 8, 6, 3, 8, False), ("act", "tanh"), ("maxpool", 6, 6, 8, 2), ("conv", 3, 3, 8, 3, 256, False),
              ("act", "relu"), ("fc", 256, 5), ("act", "softmax")], "ce_multiclass", "sgd"),
    "k257": ([("conv", 8, 8, 6, 3, 8, False), ("act", "tanh"), ("maxpool", 6, 6, 8, 2), ("conv", 3, 3, 8, 3, 257, False),
              ("act", "relu"), ("fc", 257, 5), ("act", "softmax")], "ce_multiclass", "sgd"),
    # one output channel; two activations in front, the nearer one in a phase of its own
    "k1": ([("conv", 8, 8, 6, 3, 8, False), ("act", "tanh"), ("act", "sigmoid"), ("conv", 6, 6, 8, 6, 1, False),
            ("fc", 1, 2)], "mse", "sgd"),
    # no layer between the two; rows of 392 values in 128 lanes, an uneven last range of channels
    "direct": ([("conv", 9, 9, 6, 3, 8, False), ("conv", 7, 7, 8, 7, 61, False), ("act", "tanh"), ("act", "leaky_relu", (0.1, 0.0)),
                ("fc", 61, 9), ("act", "tanh"), ("fc", 9, 3), ("act", "sigmoid")], "mse", "adam"),
    # a split net whose second convolution's gradient takes the scratch area next; one row more than a wave of pieces
    "behind": ([("conv", 14, 14, 1, 3, 6, False), ("act", "tanh"), ("conv", 12, 12, 6, 3, 16, False), ("act", "sigmoid"),
                ("avepool", 10, 10, 16, 2), ("act", "tanh"), ("conv", 5, 5, 16, 5, 20, False),
                ("fc", 20, 4)], "mse", "momentum"),
    "act_only": ([("conv", 8, 8, 2, 3, 6, False), ("act", "tanh"), ("conv", 6, 6, 6, 3, 13, False), ("act", "tanh"),
                  ("conv", 4, 4, 13, 4, 33, False), ("act", "tanh"), ("fc", 33, 4)], "mse", "adagrad"),
    # rows that are no multiple of four values
    "odd": ([("conv", 8, 8, 6, 3, 9, False), ("act", "tanh"), ("maxpool", 6, 6, 9, 2), ("conv", 3, 3, 9, 3, 12, False),
             ("act", "tanh"), ("fc", 12, 3)], "mse", "sgd"),
}


@pytest.mark.parametrize("batch", [1, 5, 90])
@pytest.mark.parametrize("name", list(HELD_NETS))
def test_filters_held_in_registers(T, O, W, name, batch):
    """Every tensor of nets with a convolution whose window is its whole input, against the oracle; two passes, so that the
    second one runs on what the first one left behind."""
    spec, params, x, t, batch, loss, kind, _, net, ref = build(T, O, W, name, batch, SAMPLE | FUSE, nets=HELD_NETS)
    xd, td = T.to_device(x), T.to_device(t)
    opt = T.opt_desc(kind, alpha=1e-3)
    net.train_step(opt, loss, batch, xd, td)
    ref.train_step(O.opt_desc(kind, alpha=1e-3), loss, x, t)
    net.train_step(None, loss, batch, xd, td, do_update=False)
    ref.train_step(O.opt_desc(kind), loss, x, t, do_update=False)
    for i, l in enumerate(spec):
        assert_close(net.layer_out(i, batch), ref.layer_out(i, batch), what=f"layer {i} output")
        assert_close(net.layer_dx(i, batch), ref.layer_dx(i, batch), what=f"layer {i} dX")
        if net.param_size(i, 0):
            assert_close(net.layer_grad(i, 0), ref.layer_dw(i), what=f"layer {i} dW")
    net.close()
