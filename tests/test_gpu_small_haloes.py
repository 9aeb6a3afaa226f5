"""Many small haloes beside a few large ones in one call: the launches are shaped by all of them
together, each halo's sums by itself alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _catalogue(sizes, seed):
    rng = np.random.default_rng(seed)
    h = np.repeat(np.arange(len(sizes)), sizes)
    x = rng.uniform(-20, 20, (len(sizes), 3))[h] + 0.004 * rng.normal(size=(len(h), 3))
    m = np.exp(rng.uniform(np.log(1e4), np.log(1e6), len(h)))
    return x.astype(np.float32), m.astype(np.float32), np.concatenate([[0], np.cumsum(sizes)])


SIZES = [[20] * 5000, [1, 0, 3, 257, 256, 255] * 700, [40] * 4200 + [9000, 1300],
         [30000] + [0, 7] * 2000]


@pytest.mark.parametrize("sizes", SIZES, ids=["equal", "edges", "last_large", "first_large"])
def test_self_sums_of_many_small_haloes(gpu, sizes):
    import torch

    from pyhalma_amd import engine

    x, m, off = _catalogue(np.array(sizes), len(sizes))
    print(f"haloes={len(sizes)} members={len(m)}", flush=True)
    S = engine.pot_sum_self(off, m, *x.T)
    bound = engine.pot_sym_error_bound()
    rng = np.random.default_rng(1)
    for h in np.unique(np.concatenate([rng.integers(0, len(sizes), 40), np.argsort(sizes)[-3:],
                                       [0, len(sizes) - 1]])):
        a, b = off[h], off[h + 1]
        if b == a:
            continue
        q = torch.from_numpy(x[a:b]).cuda().double()
        want = torch.zeros(b - a, dtype=torch.float64, device=q.device)
        mm = torch.from_numpy(m[a:b]).cuda().double()
        for i in range(0, b - a, 1000):
            d = q[i:i + 1000, None] - q[None]
            w = d.pow(2).sum(2).rsqrt()
            w[(d == 0).any(2)] = 0.0
            want[i:i + 1000] = (w * mm).sum(1)
        assert bool(((S[a:b] - want).abs() <= bound * want).all()), h
        alone = engine.pot_sum_self(np.array([0, b - a]), m[a:b], *x[a:b].T)
        assert torch.equal(alone, S[a:b]), h


@pytest.mark.parametrize("sizes", SIZES, ids=["equal", "edges", "last_large", "first_large"])
def test_softened_sums_of_many_small_haloes(gpu, sizes):
    import torch

    from pyhalma_amd import engine

    eps = 5e-4
    x, m, off = _catalogue(np.array(sizes), 7 + len(sizes))
    print(f"haloes={len(sizes)} members={len(m)}", flush=True)
    rows = torch.from_numpy(np.concatenate([x, m[:, None]], 1)).cuda()
    r = engine.pot_soft_self(off, rows, eps, pot=True, acc=True)
    one = engine.pot_soft_self(off, rows, eps, pot=True, acc=True, wsum=True)  # one-sided
    # 13u and 15u of S; 26u and 28u of the sum of |terms| of a, no term beyond 0.1 Mpc
    assert bool(((r["pot"] - one["pot"]).abs() <= 28 * 2.0 ** -24 * one["pot"]).all())
    scale = one["wsum"][:, None] * 0.1
    assert bool(((r["acc"] - one["acc"]).abs() <= 54 * 2.0 ** -24 * scale + 1e-30).all())
    rng = np.random.default_rng(1)
    for h in np.unique(np.concatenate([rng.integers(0, len(sizes), 30), np.argsort(sizes)[-3:]])):
        a, b = off[h], off[h + 1]
        alone = engine.pot_soft_self(np.array([0, b - a]), rows[a:b], eps, pot=True, acc=True)
        assert torch.equal(alone["pot"], r["pot"][a:b])
        assert torch.equal(alone["acc"], r["acc"][a:b])


@pytest.mark.parametrize("large", [0, 1, 7])
def test_many_tiny_spheres(gpu, large):
    """Spheres of no or a few points, alone and with some of thousands among them (the largest
    count decides how the hits are sorted)."""
    from scipy.spatial import cKDTree

    from pyhalma_amd import engine

    rng = np.random.default_rng(large)
    x = rng.uniform(0, 10, (60000, 3))
    c = rng.uniform(0, 10, (20000, 3))
    r = np.full(len(c), 0.08)
    r[rng.integers(0, len(c), large)] = rng.uniform(1.0, 4.5, large)
    print(f"spheres={len(c)} large={large}", flush=True)
    off, idx, mass = engine.ball_query(*x.T, c, r, m=np.ones(len(x)))
    want = [np.sort(k) for k in cKDTree(x).query_ball_point(c, r)]
    assert np.array_equal(np.diff(off), [len(k) for k in want])
    assert np.array_equal(idx.cpu().numpy(), np.concatenate(want))
    assert np.array_equal(mass, np.diff(off))


@pytest.mark.parametrize("max_iter", [2, 5, 100])
@pytest.mark.parametrize("sizes", [[20, 21] * 1500, [255, 256, 257, 63, 64, 65] * 15,
                                   [10, 11] * 300 + [2001, 3000, 500, 501]],
                         ids=["tiny", "edges", "mixed"])
def test_unbinding_of_many_small_haloes(gpu, sizes, max_iter):
    """Haloes of at most 256 members take a wavefront each for their further passes, larger ones
    a workgroup: masks and pass counts of the plain FP64 comparator, v_cm of the bound ones."""
    import torch
    from test_gpu_unbind_tail import _groups, _haloes

    from pyhalma_amd import engine

    X, V, M = _haloes(sizes, 5)
    print(f"haloes={len(sizes)} members={len(M)} max_iter={max_iter}", flush=True)
    r = engine.unbind(_groups(sizes), *X.T, *V.T, M, max_iter=max_iter, with_pot=True)
    bound, iters = engine.unbind_plain_f64(_groups(sizes), *X.T, *V.T, M, max_iter=max_iter)
    assert torch.equal(r.bound, bound)
    assert np.array_equal(r.iters.cpu().numpy(), iters)
    assert r.stats["passes"] >= iters.max()
    # the pairs of the reference's loop: every pass over the bound set it began with
    n = np.array(sizes, float)
    assert (n * n).sum() <= r.stats["pairs"] <= (n * n * iters).sum()
    if max_iter < 100:
        return
    off = np.concatenate([[0], np.cumsum(sizes)])
    b = r.bound.cpu().numpy().astype(bool)
    m = M.astype(np.float64) * b
    mass = np.add.reduceat(m, off[:-1])
    want = np.add.reduceat(m[:, None] * V.astype(np.float64), off[:-1]) / np.maximum(mass, 1e-300)[:, None]
    got = r.vcm.cpu().numpy()
    assert np.abs(got - want)[mass > 0].max() <= 1e-12 * np.abs(V).max()
