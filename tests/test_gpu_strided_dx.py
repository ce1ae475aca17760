"""dX of strided convolutions (one product per phase of the stride) against the oracle."""
import numpy as np
import pytest

from conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    # in_w, in_h, in_c, kw, kh, out_c, same, sw, sh, batch
    (45, 37, 21, 5, 5, 45, False, 2, 2, 3),   # 9, 6, 6 and 4 taps
    (6, 5, 8, 5, 5, 3, True, 2, 2, 1),        # padding, phases of a few pixels
    (12, 9, 6, 1, 1, 5, False, 2, 2, 2),      # three phases without a tap: zero gradient
    (20, 11, 33, 3, 2, 17, True, 4, 1, 2),    # four phases along x, one of them without a tap
    (9, 23, 5, 2, 3, 70, False, 1, 3, 4),     # three along y
    (16, 16, 40, 3, 3, 64, True, 2, 1, 9),    # several tiles and splits a phase
    (7, 1, 5, 3, 1, 4, True, 2, 2, 2),        # one image row: two phases have no pixel
])
def test_strided_dx_matches_oracle(T, O, cfg):
    iw, ih, ic, kw, kh, oc, same, sw, sh, bs = cfg
    opts = dict(pad_same=same, w_stride=sw, h_stride=sh)
    d, do = T.conv_desc(iw, ih, ic, kw, kh, oc, **opts), O.conv_desc(iw, ih, ic, kw, kh, oc, **opts)
    ow, oh = T.conv_out_shape(d)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((bs, ic * ih * iw)).astype(np.float32)
    w = rng.uniform(-0.3, 0.3, oc * ic * kh * kw).astype(np.float32)
    dy = rng.standard_normal((bs, oc * oh * ow)).astype(np.float32)
    dx = T.to_device(np.full(x.shape, 7, np.float32))  # every element is overwritten
    T.conv2d_bwd(d, bs, T.to_device(x), T.to_device(w), T.to_device(dy), dx, None, None)
    assert_close(dx.numpy(), O.conv2d_bwd(do, x, w, dy)[0], what="dx")
