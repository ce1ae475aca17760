"""The fully-connected forward product on its own kernel against the general one, which takes over where the input is not
aligned: the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out,batch", [
    (4096, 4096, 256),      # tiles of 128 x 128, slices
    (4100, 4092, 250),      # ... ragged, a last slice that is shorter
    (1028, 4100, 2050),     # 64 x 64, one slice, a last step of four
    (131072, 256, 64),      # tiles of 64 x 128
    (4096, 4096, 64),       # 64 x 64
    (1028, 1020, 250),      # ... ragged, a last slice that is shorter
    (5376, 1308, 278),      # 32 x 256
    (3996, 676, 94),        # 32 x 128
    (16004, 252, 33),
])
def test_same_bits_as_the_general_kernel(T, n_in, n_out, batch):
    rng = np.random.default_rng(91)
    x = rng.standard_normal((batch, n_in)).astype(np.float32)
    x[0, 3], x[batch // 2, n_in - 1] = np.inf, np.nan
    w, b = rng.uniform(-1, 1, (n_in, n_out)).astype(np.float32), rng.standard_normal(n_out).astype(np.float32)
    xd, wd, bd = T.to_device(x), T.to_device(w), T.to_device(b)
    room = T.to_device(np.concatenate([[np.float32(0)], x.ravel()]).astype(np.float32))
    aside = T.DevBuf.view(room.ptr.value + 4, (batch, n_in))
    y, want, tags = T.DevBuf((batch, n_out)), T.DevBuf((batch, n_out)), []
    for src, dst in ((xd, y), (aside, want)):
        T.profile_begin()
        T.fc_fwd(n_in, n_out, True, batch, src, wd, bd, dst)
        tags.append({r["tag"].split()[0] for r in T.profile_end()})
    assert "fc_fwd_f32" in tags[0] and "fc_fwd_gemm" in tags[1], tags
    assert np.array_equal(y.numpy(), want.numpy(), equal_nan=True)
    rows = np.setdiff1d(np.arange(batch), (0, batch // 2))
    exact = x[rows].astype(np.float64) @ w.astype(np.float64) + b
    size = np.abs(x[rows]).astype(np.float64) @ np.abs(w).astype(np.float64) + np.abs(b)
    assert (np.abs(y.numpy()[rows] - exact) <= (n_in + 2) * 2.0 ** -24 * size).all()
