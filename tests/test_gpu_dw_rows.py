"""dW and db of 3x3 windows at sizes where the filter rows are workgroups of their own (the slices of pixels leave compute
units idle) and just behind that, against float64."""
import numpy as np
import pytest

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
@pytest.mark.parametrize("w,h,ci,co,batch", [
    (15, 15, 24, 48, 37),
    (8, 3, 16, 16, 1),
    (13, 9, 33, 17, 3),     # two blocks of input channels, the second of one
    (24, 24, 16, 20, 9),    # rows of whole words
    (65, 5, 20, 40, 2),     # two column tiles
    (12, 12, 64, 64, 90),   # 90 slices of two input blocks: rows together
])
def test_weight_gradient_of_filter_rows(T, w, h, ci, co, batch, same):
    rng = np.random.default_rng(71)
    d = T.conv_desc(w, h, ci, 3, 3, co, pad_same=same)
    ow, oh = T.conv_out_shape(d)
    if ow < 1 or oh < 1:
        pytest.skip("no output")
    x = rng.standard_normal((batch, ci, h, w)).astype(np.float32)
    dy = rng.standard_normal((batch, co, oh, ow)).astype(np.float32)
    dw, db = T.DevBuf((co, ci, 3, 3)), T.DevBuf((co,))
    T.conv2d_bwd(d, batch, T.to_device(x), T.to_device(rng.standard_normal(dw.shape).astype(np.float32)), T.to_device(dy), None, dw, db)
    want_w, want_b, size_w, size_b = conv_grad64(x, dy, 1 if same else 0)
    n = batch * ow * oh   # (sums of n rounded products, in any order)
    assert (np.abs(dw.numpy() - want_w) <= (n + 1) * 2.0 ** -24 * size_w).all()
    assert (np.abs(db.numpy() - want_b) <= (n + 1) * 2.0 ** -24 * size_b).all()
