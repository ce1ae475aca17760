"""dX and dW of a convolution of any window where one call computes both: dW's launch packs dX's filters and dX's launch adds up
dW's slices. Bit for bit what the two give one at a time, which tests/test_gpu_conv_any.py compares with the oracle."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def layer(T, wd, ht, ic, oc, k, st, same, bs):
    rng = np.random.default_rng(3)
    d = T.conv_desc(wd, ht, ic, k, k, oc, pad_same=same, w_stride=st, h_stride=st)
    ow, oh = ((-(-n // st)) if same else (-(-(n - k + 1) // st)) for n in (wd, ht))
    x = T.to_device(rng.standard_normal((bs, ic * ht * wd)).astype(np.float32))
    w = T.to_device(rng.standard_normal(oc * ic * k * k).astype(np.float32))
    dy = T.to_device(rng.standard_normal((bs, oc * oh * ow)).astype(np.float32))
    return d, x, w, dy


@pytest.mark.parametrize("cfg", [
    # width, height, in_c, out_c, window, stride, same, batch: the launches that this road leaves out
    ((45, 37, 21, 45, 5, 2, False, 19), {"conv_any_pack", "conv_dw_splitk_reduce"}),
    ((23, 19, 5, 7, 5, 2, True, 64), None),       # (another road)
    ((31, 29, 6, 18, 7, 1, False, 40), {"conv_any_pack", "conv_dw_splitk_reduce"}),
    ((40, 33, 70, 66, 5, 2, False, 4), {"conv_any_pack"}),     # several tiles of channels in either direction, sums apart
    ((64, 61, 3, 33, 7, 2, True, 128), {"conv_any_pack", "conv_dw_splitk_reduce"}),     # many slices
])
@pytest.mark.parametrize("with_db", [True, False])
def test_together_as_one_by_one(T, cfg, with_db):
    (wd, ht, ic, oc, k, st, same, bs), without = cfg
    d, x, w, dy = layer(T, *cfg[0])
    both, single = ([T.DevBuf((bs, ic * ht * wd)), T.DevBuf((oc * ic * k * k,)), T.DevBuf((oc,)) if with_db else None]
                    for _ in range(2))
    T.profile_begin()
    T.conv2d_bwd(d, bs, x, w, dy, *both)
    tags = [e["tag"].split()[0] for e in T.profile_end()]
    packs_or_adds = {"conv_any_pack", "conv_dw_splitk_reduce"}
    if without is None:
        assert not {"conv_dx_any_x3", "conv_dw_any", "conv_dw_db_any"} & set(tags), tags
    else:
        assert "conv_dx_any_x3" in tags and packs_or_adds & set(tags) == packs_or_adds - without, tags
    T.conv2d_bwd(d, bs, x, w, dy, single[0], None, None)
    T.conv2d_bwd(d, bs, x, w, dy, None, single[1], single[2])
    for a, b, name in zip(both, single, ("dx", "dw", "db")):
        assert a is None or np.array_equal(a.numpy(), b.numpy()), name


def test_together_no_slower_than_one_by_one(T):
    """dW's workgroups are whole rounds of the chip, and the packing's must not come in between: the last of dW's then run in a
    round of their own (155 x 1862 weights over 54 images: 186 us a call instead of 134; one by one 137)."""
    (ic, oc, k, ht, wd, bs) = (38, 155, 7, 50, 13, 54)
    d, x, w, dy = layer(T, wd, ht, ic, oc, k, 2, False, bs)
    dx, dw, db = T.DevBuf((bs, ic * ht * wd)), T.DevBuf((oc * ic * k * k,)), T.DevBuf((oc,))

    def us(call):
        best = np.inf
        for _ in range(8):
            T.sync()
            start = time.perf_counter()
            for _ in range(20):
                call()
            T.sync()
            best = min(best, (time.perf_counter() - start) / 20 * 1e6)
        return best

    together = us(lambda: T.conv2d_bwd(d, bs, x, w, dy, dx, dw, db))
    one_by_one = us(lambda: (T.conv2d_bwd(d, bs, x, w, dy, dx, None, None), T.conv2d_bwd(d, bs, x, w, dy, None, dw, db)))
    # (in between, 1.36 times; behind, 0.98 times)
    assert together < 1.15 * one_by_one, (together, one_by_one)
