"""Group reductions at the edges of their workgroup sizes, density peaks at the edges
between grid nodes and cell statistics at the edges of a wavefront's cell, on the GPU.

Sums are double-double rounded once: M within a unit of the exactly rounded sum, the centre
and the mean velocity (quotients of two) within three; bounding boxes exact; the radius two
rounded squares, their sums and a root of exact differences, within 4 units of the one from
the returned centre.  Density peaks are equal to the oracle's, cleaning as in its own tests."""
import math

import numpy as np
import pytest
import torch

import oracle
from test_gpu_cleaning import _check, _dev_groups

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1025, 2, 4095, 4096, 4097, 9000, 5]


def _groups():
    off = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int64)
    mem = np.random.default_rng(8).permutation(int(off[-1]) + 100)[:off[-1]].astype(np.int32)
    return mem, [np.sort(mem[off[k]:off[k + 1]]) for k in range(len(SIZES))]


@pytest.mark.parametrize("pt,mt", [(np.float32, np.float32), (np.float64, np.float64),
                                   (np.float32, np.float64)])
def test_reduce_at_the_workgroup_edges(gpu, pt, mt):
    from pyhalma_amd import engine

    rng = np.random.default_rng(9)
    mem, groups = _groups()
    n = len(mem) + 100
    pos = [(a + rng.uniform(1, 5, n)).astype(pt) for a in (0, 30, 4)]
    vel = [rng.uniform(50, 300, n).astype(pt) for _ in range(3)]
    m = rng.uniform(1, 9, n).astype(mt)
    out = engine.group_reduce(_dev_groups(groups), *pos, m, *vel).cpu().numpy()
    u = 2.0 ** -52
    p64, v64, m64 = [a.astype(np.float64) for a in pos], [a.astype(np.float64) for a in vel], \
        m.astype(np.float64)
    for k, g in enumerate(groups):
        M = math.fsum(m64[g])
        np.testing.assert_allclose(out[k, 0], M, rtol=u, atol=0)
        for d in range(3):
            np.testing.assert_allclose(out[k, 1 + d], math.fsum(m64[g] * p64[d][g]) / M, rtol=3 * u)
            np.testing.assert_allclose(out[k, 4 + d], math.fsum(m64[g] * v64[d][g]) / M, rtol=3 * u)
            assert out[k, 8 + d] == p64[d][g].min() and out[k, 11 + d] == p64[d][g].max()
        r = max(math.sqrt(sum((out[k, 1 + d] - p64[d][i]) ** 2 for d in range(3))) for i in g)
        np.testing.assert_allclose(out[k, 7], r, rtol=4 * u)
        np.testing.assert_allclose(out[k, 14], M, rtol=2e-12)


@pytest.mark.parametrize("shift,ll", [(0.0, 0.1), (3e5, 1e-3), (-7.0, 0.0)])
def test_peak_between_the_nodes(gpu, shift, ll):
    from pyhalma_amd import engine

    # members at the midpoints of neighbouring nodes and a few units either side
    rng = np.random.default_rng(10)
    lo, hi = shift - 1.0, shift + 1.0
    nodes = np.linspace(lo - ll, hi + ll, 50)
    mid = 0.5 * (nodes[1:-2] + nodes[2:-1])
    mid = mid[(mid > lo) & (mid < hi)]
    n = 3000
    pos = []
    for _ in range(3):
        v = rng.choice(mid[:9], n)
        for _ in range(3):
            v = np.where(rng.random(n) < 0.5, np.nextafter(v, rng.choice([-1e9, 1e9], n)), v)
        v[0], v[1] = lo, hi
        pos.append(v)
    m = rng.integers(1, 4, n).astype(np.float64)
    grp = np.arange(n)
    got = engine.density_peak(_dev_groups([grp, grp[:40]]), *pos, m, ll).cpu().numpy()
    assert tuple(got[0]) == oracle.density_peak(grp, *pos, m, ll)
    assert tuple(got[1]) == oracle.density_peak(grp[:40], *pos, m, ll)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_cells_at_the_wavefront_edges(gpu, dtype):
    from pyhalma_amd import engine

    # one group per cell size: a tight cell of that many members and a spread of loners
    rng = np.random.default_rng(11)
    P, V, groups, base = [], [], [], 0
    for h, c in enumerate([1, 2, 3, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1400]):
        p = np.concatenate([rng.uniform(-1e-3, 1e-3, (c, 3)), rng.uniform(-8, 8, (30, 3))])
        v = rng.normal(size=(c + 30, 3)) * 40
        v[:max(c // 12, 1), 0] += 400.0
        P.append(p + 100.0 * h)
        V.append(v)
        groups.append(np.arange(base, base + c + 30))
        base += c + 30
    P, V = np.concatenate(P).astype(dtype), np.concatenate(V).astype(dtype)
    M = rng.uniform(0.5, 2, base).astype(dtype)
    args = (P[:, 0], P[:, 1], P[:, 2], V[:, 0], V[:, 1], V[:, 2], M)
    res = engine.phase_space_clean(_dev_groups(groups), *args, 1.0, 1.0, 3.0, min_part=0, minp=1)
    per, kept = oracle.phase_space_clean(groups, *args, 1.0, 1.0, 3.0, min_part=0, minp=1)
    _check(res, per, kept)
