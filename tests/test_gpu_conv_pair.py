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
