"""Workspace sizes follow the data and not a limit the caller passes (host queries, no GPU)."""
import ctypes

import numpy as np


def _off(*sizes):
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    return len(sizes), off.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), off


def test_refine_centres_workspace_is_free_of_the_iteration_limit():
    from pyhalma_amd import _lib

    size = _lib.load().halma_refine_centres_workspace_size
    H, off, _keep = _off(3000, 0, 100000)
    for limit in (0, 1, 200, 10 ** 6, 2 ** 31 - 2, 2 ** 31 - 1):
        assert size(H, off, limit) == size(H, off, 4) > 0


def test_soft_self_workspace_is_bounded():
    """The slots of the symmetric form: 4 GiB at most, also for the largest halo it takes and
    for the smallest that it leaves to the one-sided form, which needs tens of bytes a member."""
    from pyhalma_amd import _lib

    size = _lib.load().halma_soft_self_workspace_size
    for sizes in ([1 << 20], [1 << 21], [(1 << 21) + 1], [1 << 22], [1 << 23],
                  [1 << 21, 1 << 23, 1 << 21, 100], [200000] * 20):
        H, off, _keep = _off(*sizes)
        assert 0 < size(H, off) <= (4 << 30) + 200 * sum(sizes), sizes
