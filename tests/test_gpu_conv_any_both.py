"""dX and dW of a convolution of any window where one call computes both: dW's launch packs dX's filters and dX's launch adds up
dW's slices. Bit for bit what the two give one at a time, which tests/test_gpu_conv_any.py compares with the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    # width, height, in_c, out_c, window, stride, same, batch: True where this road is known to be taken
    ((45, 37, 21, 45, 5, 2, False, 19), True),
    ((23, 19, 5, 7, 5, 2, True, 64), None),
    ((31, 29, 6, 18, 7, 1, False, 40), None),
    ((40, 33, 70, 66, 5, 2, False, 4), None),     # several tiles of channels in either direction, sums apart
    ((64, 61, 3, 33, 7, 2, True, 128), None),     # many slices
])
@pytest.mark.parametrize("with_db", [True, False])
def test_together_as_one_by_one(T, cfg, with_db):
    (wd, ht, ic, oc, k, st, same, bs), along = cfg
    rng = np.random.default_rng(3)
    d = T.conv_desc(wd, ht, ic, k, k, oc, pad_same=same, w_stride=st, h_stride=st)
    ow, oh = ((-(-n // st)) if same else (-(-(n - k + 1) // st)) for n in (wd, ht))
    x = T.to_device(rng.standard_normal((bs, ic * ht * wd)).astype(np.float32))
    w = T.to_device(rng.standard_normal(oc * ic * k * k).astype(np.float32))
    dy = T.to_device(rng.standard_normal((bs, oc * oh * ow)).astype(np.float32))
    both, single = ([T.DevBuf((bs, ic * ht * wd)), T.DevBuf((oc * ic * k * k,)), T.DevBuf((oc,)) if with_db else None]
                    for _ in range(2))
    T.profile_begin()
    T.conv2d_bwd(d, bs, x, w, dy, *both)
    tags = [e["tag"].split()[0] for e in T.profile_end()]
    if along:
        assert "conv_dx_any_x3" in tags and not {"conv_any_pack", "conv_dw_splitk_reduce"} & set(tags), tags
    T.conv2d_bwd(d, bs, x, w, dy, single[0], None, None)
    T.conv2d_bwd(d, bs, x, w, dy, None, single[1], single[2])
    for a, b, name in zip(both, single, ("dx", "dw", "db")):
        assert a is None or np.array_equal(a.numpy(), b.numpy()), name
