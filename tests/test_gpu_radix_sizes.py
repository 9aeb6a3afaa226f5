"""Group lists from labels through the radix sort at the edges of its tiles: sizes around
1024, 4096 and 2^20 keys (where the tile size changes), labels few and many, sorted and
shuffled: members ascending within a group, groups by smallest member; a
sort of fewer keys than its workspace was sized for."""
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


def test_sort_of_fewer_keys_than_its_workspace(gpu):
    """A sphere query's workspace holds the sort of all its points in large tiles; one sphere
    with 2^20 - 1 of them sorts its hits in small tiles, whose tables are four times longer."""
    from pyhalma_amd import engine

    n, hits = (1 << 20) + 5000, (1 << 20) - 1
    rng = np.random.default_rng(1)
    x = rng.uniform(-0.5, 0.5, (n, 3))
    inside = np.zeros(n, bool)
    inside[rng.permutation(n)[:hits]] = True
    x[~inside] += 5.0
    print(f"points={n} hits={hits}", flush=True)
    off, idx, _ = engine.ball_query(*x.T, [[0.0, 0.0, 0.0]], [1.0])
    assert list(off) == [0, hits]
    assert np.array_equal(idx.cpu().numpy(), np.nonzero(inside)[0])
