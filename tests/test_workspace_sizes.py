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
