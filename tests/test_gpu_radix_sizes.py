"""Group lists from labels through the radix sort at the edges of its tiles: sizes around
1024, 4096 and 2^20 keys (where the tile size changes), labels few and many, sorted and
shuffled: members ascending within a group, groups by smallest member."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 255, 257, 1023, 1024, 1025, 4095, 4097, 65537,
                               (1 << 20) - 1, 1 << 20, (1 << 20) + 4097])
@pytest.mark.parametrize("groups", [1, 300, 0])
def test_groups_of_sorted_labels(gpu, n, groups):
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(n + groups)
    k = groups if groups else n
    g = rng.integers(0, k, n)
    # a label is the group's smallest member
    first = np.full(k, n, np.int64)
    np.minimum.at(first, g, np.arange(n))
    lab = first[g].astype(np.int32)
    print(f"n={n} groups={k}", flush=True)
    r = engine.groups_from_labels(torch.from_numpy(lab).cuda(), 1)
    order = np.argsort(lab, kind="stable")
    uniq, cnt = np.unique(lab, return_counts=True)
    assert np.array_equal(r.members[: r.n_members].cpu().numpy(), order)
    assert np.array_equal(r.offsets_host, np.concatenate([[0], np.cumsum(cnt)]))


def test_sort_workspace_holds_every_smaller_sort():
    # on the host: the tables of a sort of up to n pairs fit the workspace of n pairs
    def need(n, small=1024, large=4096):
        nb = -(-n // (large if n >= 1 << 20 else small))
        return 2 * 256 * 4 * nb + 8 * n

    def given(n):
        nb = max(-(-n // (4096 if n >= 1 << 20 else 1024)), -(-min(n, (1 << 20) - 1) // 1024))
        return 2 * 256 * 4 * nb + 8 * n

    for n in (1 << 20, (1 << 20) + 1, 1200000, 5000000):
        for m in (n, (1 << 20) - 1, 1 << 20, 1000):
            assert need(m) <= given(n)
