"""dW and db of 3x3 windows at sizes where the filter rows are workgroups of their own (the slices of pixels leave compute
units idle) and just behind that, against float64."""
import numpy as np
import pytest

from test_gpu_conv_any import within_fp32_sum

pytestmark = pytest.mark.gpu


def conv_grad64(x, dy, pad):
    x = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    dy, (oh, ow) = dy.astype(np.float64), dy.shape[2:]
    parts = {(r, s): x[:, :, r:r + oh, s:s + ow] for r in range(3) for s in range(3)}

    def dw(of):
        taps = [np.tensordot(of(dy), of(parts[r, s]), ((0, 2, 3), (0, 2, 3))) for r in range(3) for s in range(3)]
        return np.stack(taps, -1).reshape(dy.shape[1], x.shape[1], 3, 3)

    return dw(np.asarray), dy.sum((0, 2, 3)), dw(np.abs), np.abs(dy).sum((0, 2, 3))


@pytest.mark.parametrize("same", [True, False])
@pytest.mark.parametrize("w,h,ci,co,batch,kernel", [
    (15, 15, 24, 48, 37, "conv_dw_db_rows"),
    (10, 10, 33, 40, 40, "conv_dw_db_rows"),    # tiles of 8 columns; two blocks of input channels, the second of one
    (15, 15, 33, 17, 20, "conv_dw_db_rows"),    # 32 output channels a workgroup; two blocks of input channels
    (18, 15, 70, 33, 13, "conv_dw_db_rows"),    # three of them, a block of output channels of one
    (26, 24, 16, 20, 9, "conv_dw_db_rows"),     # tiles of 32 columns
    (33, 20, 30, 36, 8, "conv_dw_db_rows"),     # ... and, padded, two of them
    (50, 12, 18, 30, 6, "conv_dw_db_rows"),     # tiles of 64 columns
    (66, 9, 20, 40, 6, "conv_dw_db_rows"),      # ... and, padded, two of them
    (12, 12, 64, 64, 90, "conv_dw_db_halo"),    # 90 slices of two input blocks: rows together
])
def test_weight_gradient_of_filter_rows(T, w, h, ci, co, batch, kernel, same):
    rng = np.random.default_rng(71)
    d = T.conv_desc(w, h, ci, 3, 3, co, pad_same=same)
    ow, oh = T.conv_out_shape(d)
    x = rng.standard_normal((batch, ci, h, w)).astype(np.float32)
    dy = rng.standard_normal((batch, co, oh, ow)).astype(np.float32)
    dw, db = T.DevBuf((co, ci, 3, 3)), T.DevBuf((co,))
    xd, wd, dyd = T.to_device(x), T.to_device(rng.standard_normal(dw.shape).astype(np.float32)), T.to_device(dy)
    T.profile_begin()
    T.conv2d_bwd(d, batch, xd, wd, dyd, None, dw, db)
    tags = {e["tag"].split()[0] for e in T.profile_end()}
    assert kernel in tags, tags
    want_w, want_b, size_w, size_b = conv_grad64(x, dy, 1 if same else 0)
    n = batch * ow * oh
    for got, want, size, name in ((dw.numpy(), want_w, size_w, "dw"), (db.numpy(), want_b, size_b, "db")):
        # n terms in order, each addition rounding to 2^-24 of a partial sum that grows as a random walk, leave 2^-24 sqrt(n / 6)
        # of the result, a product's own rounding less than 2^-24 of it; in slices that are added it is less
        assert np.linalg.norm(got - want) <= 2 ** -24 * (2 + np.sqrt(n / 6)) * np.linalg.norm(want), name
        assert within_fp32_sum(got, want, size), name
