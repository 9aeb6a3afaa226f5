"""Progenitors of haloes whose members end within, at and past a thread's batch, on the GPU
(equal to the oracle)."""
import numpy as np
import pytest

from test_gpu_progenitors import _both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", [1, 10 ** 9])
def test_members_at_the_batch_edges(gpu, spread):
    # batches of 8 x 512 members; the last members alone have a progenitor of their own
    rng = np.random.default_rng(7)
    sizes = [1, 2, 511, 512, 513, 4095, 4096, 4097, 4609, 8192, 8193]
    ids = rng.permutation(np.arange(sum(sizes) + 50, dtype=np.int64)) * spread - 1000
    new = np.split(ids[:sum(sizes)], np.cumsum(sizes)[:-1])
    old = [h[:-1] for h in new if len(h) > 1] + [h[-1:] for h in new] + [ids[sum(sizes):]]
    got, want = _both(new, rng.uniform(1, 100, len(new)), old, rng.uniform(1, 100, len(old)))
    assert got == want
