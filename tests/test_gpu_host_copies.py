"""Copies between host memory and the device around the sizes at which their path changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 16, 4097, 16 * 1024, 16 * 1024 + 1, 64 * 1024 - 1, 64 * 1024, 64 * 1024 + 1])
def test_bytes_survive_the_round_trip(T, n):
    rng = np.random.default_rng(n)
    for offset in (0, 1, 4):
        a = rng.integers(0, 256, n, dtype=np.uint8)
        buf = T.DevBuf((n + 32,), np.uint8).upload(np.zeros(n + 32, np.uint8))
        at = T.DevBuf.view(buf.ptr.value + offset, (n,), np.uint8)
        at.upload(a)
        assert np.array_equal(at.numpy(), a)
        around = buf.numpy()
        assert not around[:offset].any() and not around[offset + n:].any()


def test_a_source_may_be_overwritten_at_once_and_the_ring_comes_round(T):
    a = np.empty(1000, np.float32)
    bufs = [T.DevBuf(a.shape) for _ in range(50)]
    for i, b in enumerate(bufs):
        a[:] = i
        b.upload(a)
    for i, b in enumerate(bufs):
        assert (b.numpy() == i).all()


@pytest.mark.parametrize("n", [1 << 13, 1 << 14])
def test_a_copy_past_the_end_of_its_allocation_is_an_error(T, n):
    buf = T.DevBuf((n,), np.uint8).upload(np.arange(n, dtype=np.uint8))
    a = np.zeros(n, np.uint8)
    for first in (1, n // 2, n - 1):
        view = T.DevBuf.view(buf.ptr.value + first, (n,), np.uint8)
        with pytest.raises(T.TdhError, match="past the end of its allocation"):
            view.upload(a)
        with pytest.raises(T.TdhError, match="past the end of its allocation"):
            view.numpy()
    assert np.array_equal(buf.numpy(), np.arange(n, dtype=np.uint8))
