"""Several arrays to the device in one transfer: the same tensors as one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [None, np.float32, np.float64])
@pytest.mark.parametrize("big", [0, 1 << 18, (1 << 18) + 1, 1 << 20])
def test_packed_like_single(gpu, dtype, big):
    import torch

    from pyhalma_amd import device

    rng = np.random.default_rng(3)
    arrays = [rng.random(5).astype(np.float32), np.zeros(0), rng.integers(0, 9, 7),
              rng.random((4, 6))[:, ::2], rng.integers(0, 2, 3).astype(np.uint8),
              torch.arange(4), rng.random(big).astype(np.float32), rng.random(1)]
    if dtype is not None:
        arrays += [np.arange(3, dtype=">f8"), [1, 2, 3]]  # numpy converts these
    got = device.to_dev_all(arrays, dtype)
    for a, t in zip(arrays, got):
        want = device.to_dev(a, dtype)
        assert t.dtype == want.dtype and t.shape == want.shape and t.is_contiguous()
        assert t.device == want.device and torch.equal(t, want)
    assert device.to_dev_all([]) == []
    for t in device.to_dev_all([np.zeros((0, 3)), np.zeros(0, np.int64)], dtype):
        assert t.numel() == 0 and t.is_cuda
