"""dW of fully-connected layers in three parts against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("n_in,n_out,batch", [
    (1024, 1024, 1024),
    (4096, 4096, 384),      # the fewest samples, one slice
    (1020, 1028, 515),      # ragged on every side, a last step of three samples
    (64, 8192, 1500),       # tiles of 64 inputs, slices of samples
    (8200, 64, 1037),       # tiles of 64 outputs
])
def test_weight_gradient(T, n_in, n_out, batch, accumulate):
    rng = np.random.default_rng(81)
    x = rng.standard_normal((batch, n_in)).astype(np.float32)
    x[:, ::3] = np.maximum(x[:, ::3], 0)
    x[:, 5] = 0
    dy = rng.standard_normal((batch, n_out)).astype(np.float32)
    before = rng.standard_normal((n_in, n_out)).astype(np.float32)
    dw = T.to_device(before)
    T.profile_begin()
    T.fc_bwd(n_in, n_out, False, batch, T.to_device(x), dw, T.to_device(dy), None, dw, None, accumulate=accumulate)
    assert any(r["tag"].startswith("fc_dw_x3 ") for r in T.profile_end())
    import torch
    x, dy = torch.from_numpy(x).double(), torch.from_numpy(dy).double()
    want, size = x.T @ dy, x.abs().T @ dy.abs()
    if accumulate:
        want, size = want + torch.from_numpy(before), size + torch.from_numpy(before).abs()
    # a product loses under 2^-23 of itself, and steps of 32 samples add up in fp32 (slices and the prior value with them)
    bound = 2.0 ** -24 * (2 + 2 + batch / 32 + 8) * size
    got = torch.from_numpy(dw.numpy()).double()
    assert ((got - want).abs() <= bound).all()
    assert (got[5] == (torch.from_numpy(before).double()[5] if accumulate else 0)).all()


@pytest.mark.parametrize("value", [np.inf, np.nan, 3e38])
def test_exceptional_weight_gradient(T, value):
    rng = np.random.default_rng(82)
    n_in, n_out, batch = 1024, 1024, 390
    x, dy = (rng.standard_normal((batch, n)).astype(np.float32) for n in (n_in, n_out))
    x[3, 7], x[389, 1023] = value, -value
    dw = T.DevBuf((n_in, n_out))
    T.fc_bwd(n_in, n_out, False, batch, T.to_device(x), dw, T.to_device(dy), None, dw, None)
    got = dw.numpy()
    with np.errstate(all="ignore"):
        want = (x.astype(np.float64).T @ dy.astype(np.float64))
        fits = np.abs(want) <= np.finfo(np.float32).max
    assert (np.isnan(got) == np.isnan(want)).all()
    assert (np.isfinite(got) == fits).all()
    rows = np.setdiff1d(np.arange(n_in), (7, 1023))
    assert np.abs(got[rows] - want[rows]).max() <= 2.0 ** -24 * 24 * (np.abs(x[:, rows]).T @ np.abs(dy)).max()


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("n_in,n_out,batch,slices", [
    (4096, 4096, 256, True),
    (3000, 3000, 100, True),       # the last 1024 sums and the last 32 columns in part
    (2052, 4100, 130, False),      # dX on the fp32 kernel
    (4096, 4096, 63, False),       # too few outputs for the sums of this form
    (4096, 2050, 96, False),       # rows that dX cannot read by words
])
def test_sums_in_the_weight_gradients_launch(T, n_in, n_out, batch, slices, accumulate):
    """dX and dW of one call: dW's launch adds up dX's slices and the columns of dY. The bits of each by itself, and the bias
    gradient's error (the additions of its column)."""
    rng = np.random.default_rng(83)
    x, w, dy = (T.to_device(rng.standard_normal(s).astype(np.float32)) for s in ((batch, n_in), (n_in, n_out), (batch, n_out)))
    before = [rng.standard_normal(s).astype(np.float32) for s in ((n_in, n_out), (n_out,))]
    dw, db, alone = T.to_device(before[0]), T.to_device(before[1]), T.to_device(before[0])
    dx, single = T.DevBuf((batch, n_in)), T.DevBuf((batch, n_in))
    T.profile_begin()
    T.fc_bwd(n_in, n_out, True, batch, x, w, dy, dx, dw, db, accumulate=accumulate)
    tags = [r["tag"].split()[0] for r in T.profile_end()]
    assert ("fc_dw_direct_sums" in tags) == slices and "bias_grad_colsum" not in tags, tags
    T.fc_bwd(n_in, n_out, True, batch, x, w, dy, single, None, None)
    T.fc_bwd(n_in, n_out, False, batch, x, w, dy, None, alone, None, accumulate=accumulate)
    assert np.array_equal(dx.numpy(), single.numpy())
    assert np.array_equal(dw.numpy(), alone.numpy())
    d, prior = dy.numpy().astype(np.float64), before[1].astype(np.float64) * accumulate
    assert (np.abs(db.numpy() - (d.sum(0) + prior)) <= 2.0 ** -24 * (batch + 2) * (np.abs(d).sum(0) + np.abs(prior))).all()
