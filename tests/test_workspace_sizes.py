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


def test_sort_workspaces_never_shrink():
    """Callers size for their largest input and sort fewer: the tables of the small tiles just
    under 2^20 keys are longer than those of the large tiles from there on."""
    from pyhalma_amd import _lib

    L = _lib.load()
    sizes = [1, 1000, 1 << 19, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 1200000, 1 << 21, 5000000]
    for query in (lambda n: L.halma_fof_workspace_size(n, 0),
                  lambda n: L.halma_clean_workspace_size(n),
                  lambda n: L.halma_ball_query_workspace_size(1000, 1, n)):
        got = [query(n) for n in sizes]
        assert got[0] > 0 and got == sorted(got)
    # the tables of the small tiles (1024 keys, 256 counts and offsets a tile) within a size
    # that is otherwise proportional
    per = lambda n: L.halma_ball_query_workspace_size(1000, 1, n) / n  # noqa: E731
    assert per(1 << 20) >= 0.999 * per((1 << 20) - 1)
