"""The passes a workgroup takes by itself (haloes of at most 4096 members, while no larger one
is active) against the launched passes: the same haloes alone and beside a larger one give
the same masks, pass counts and v_cm, and those of the plain FP64 comparator; sizes around
the 64-lane, 512-thread and 4096-member edges, pass limits, fly-apart pairs that take tens
of passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _haloes(sizes, seed):
    """Virial Plummer spheres; every other one a pair of halves flying apart."""
    from pyhalma_amd import synth

    rng = np.random.default_rng(seed)
    X, V, M = [], [], []
    for k, n in enumerate(sizes):
        a = 0.005 * (max(n, 2) / 2e4) ** (1 / 3)
        m = np.exp(rng.uniform(np.log(1e4), np.log(1e6), n))
        x = synth.plummer_positions(rng, n, a)
        v = rng.normal(scale=synth.plummer_sigma1d(m.sum(), a), size=(n, 3))
        if k % 2:
            side = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)[:, None]
            x = x + side * a * np.array([1.0, 0.3, 0.2])
            v = v + side * rng.uniform(0.4, 1.2) * np.sqrt(synth.G * m.sum() / a) * np.array(
                [1.0, 0.0, 0.0])
        X.append(x + rng.uniform(-20, 20, 3))
        V.append(v)
        M.append(m)
    return (np.concatenate(X).astype(np.float32), np.concatenate(V).astype(np.float32),
            np.concatenate(M).astype(np.float32))


def _groups(sizes):
    import torch

    from pyhalma_amd import engine

    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(off[-1])
    return engine.Groups(torch.arange(n, dtype=torch.int32, device="cuda"),
                         torch.from_numpy(off).cuda(), off)


@pytest.mark.parametrize("max_iter", [1, 2, 3, 7, 100])
def test_unbind_tail_matches_launched_passes(gpu, max_iter):
    import torch

    from pyhalma_amd import engine

    small = [1, 2, 63, 64, 65, 511, 512, 513, 1000, 1001, 2000, 2001, 4095, 4096, 3000, 900]
    sizes = small + [4097]
    X, V, M = _haloes(sizes, 17)
    n = sum(small)
    print(f"max_iter={max_iter} members={len(M)}", flush=True)
    with_large = engine.unbind(_groups(sizes), *X.T, *V.T, M, max_iter=max_iter, with_pot=True)
    r = engine.unbind(_groups(small), *X[:n].T, *V[:n].T, M[:n], max_iter=max_iter,
                      with_pot=True)
    H = len(small)
    assert torch.equal(r.bound, with_large.bound[:n])
    assert torch.equal(r.iters, with_large.iters[:H])
    # double-double sums rounded to FP64: an ulp between orders at most
    assert float((r.vcm - with_large.vcm[:H]).abs().max()) <= 1e-12 * float(r.vcm.abs().max())
    # every S kept is within 1e-6 of FP64
    fin = torch.isfinite(r.pot)
    assert torch.equal(fin, torch.isfinite(with_large.pot[:n]))
    d = (r.pot[fin] - with_large.pot[:n][fin]).abs()
    assert float((d / with_large.pot[:n][fin].clamp(min=1e-300)).max()) <= 2e-6
    assert r.stats["passes"] <= max_iter
    bound, iters = engine.unbind_plain_f64(_groups(small), *X[:n].T, *V[:n].T, M[:n],
                                           max_iter=max_iter)
    assert torch.equal(r.bound, bound)
    assert np.array_equal(r.iters.cpu().numpy(), iters)
