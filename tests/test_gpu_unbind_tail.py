"""The passes a workgroup takes by itself (haloes of at most 4096 members, while no larger one
is active) against the launched passes: the same haloes alone and beside a larger one that
stays active longer than all of them (so that every pass is a launched one, which the
launch counts show) give the same masks, pass counts and v_cm, those of the plain FP64
comparator, and S within 1e-6 of FP64; sizes around the 64-lane, 512-thread and 4096-member
edges, pass limits, fly-apart pairs that take tens of passes."""
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


PEEL = 45  # passes of the halo below that remove a member


def _peeling_halo():
    """5000 members at rest and, 1 Mpc away, a chain of PEEL fast ones that loses its first
    link each pass: link k is bound by both neighbours (and those behind) and not by those
    behind alone."""
    from pyhalma_amd import synth

    rng = np.random.default_rng(4)
    n, m, d = 5000, 1e9, 1e-4
    core = synth.plummer_positions(rng, n, 0.05)
    core *= np.minimum(1.0, 0.3 / np.linalg.norm(core, axis=1))[:, None]
    k = np.arange(PEEL)
    chain = 1 / np.sqrt(3) + (k * d / np.sqrt(3))[:, None] + np.zeros((1, 3))
    s_core = (m / np.linalg.norm(chain[:, None] - core[None], axis=2)).sum(1)
    behind = np.array([(1.0 / np.arange(1, PEEL - j)).sum() for j in k])
    v = np.sqrt(2 * synth.G * (s_core + m / d * (0.5 + behind)))  # E = v^2 / 2 - G S
    vel = np.zeros((n + PEEL, 3))
    vel[n:, 2] = np.where(k % 2 == 0, v, -v)
    return (np.concatenate([core, chain]).astype(np.float32), vel.astype(np.float32),
            np.full(n + PEEL, m, np.float32))


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
    X, V, M = _haloes(small, 17)
    n = sum(small)
    LX, LV, LM = _peeling_halo()
    sizes = small + [len(LM)]
    print(f"max_iter={max_iter} members={n} + {len(LM)}", flush=True)
    with_large = engine.unbind(_groups(sizes), *np.concatenate([X, LX]).T,
                               *np.concatenate([V, LV]).T, np.concatenate([M, LM]),
                               max_iter=max_iter, with_pot=True)
    r = engine.unbind(_groups(small), *X.T, *V.T, M, max_iter=max_iter, with_pot=True)
    most = int(r.iters.max())
    # one launched pass each beside the large halo, several in a workgroup without it
    assert int(with_large.iters[-1]) == min(max_iter, PEEL + 1) >= most
    assert with_large.stats["sym_launches"] >= min(max_iter, PEEL + 1)
    if max_iter > 3:
        assert r.stats["sym_launches"] < most
    H = len(small)
    assert torch.equal(r.bound, with_large.bound[:n])
    assert torch.equal(r.iters, with_large.iters[:H])
    # double-double sums rounded to FP64: an ulp between orders at most
    assert float((r.vcm - with_large.vcm[:H]).abs().max()) <= 1e-12 * float(r.vcm.abs().max())
    # every S kept is within 1e-6 of FP64 (below)
    fin = torch.isfinite(r.pot)
    assert torch.equal(fin, torch.isfinite(with_large.pot[:n]))
    d = (r.pot[fin] - with_large.pot[:n][fin]).abs()
    assert float((d / with_large.pot[:n][fin].clamp(min=1e-300)).max()) <= 2e-6
    assert r.stats["passes"] <= max_iter
    if max_iter > most:  # done: S is over the members that are bound
        off = np.concatenate([[0], np.cumsum(small)])
        for h in range(H):
            b = off[h] + torch.nonzero(r.bound[off[h]:off[h + 1]]).flatten().cpu().numpy()
            x = torch.from_numpy(X[b]).cuda().double()
            dx = x[:, None] - x[None]
            w = 1.0 / dx.pow(2).sum(2).sqrt()
            w[(dx == 0).any(2)] = 0.0
            S = (w * torch.from_numpy(M[b]).cuda().double()[None]).sum(1)
            for got in (r.pot[b], with_large.pot[b]):
                assert bool(((got - S).abs() <= 1e-6 * S).all()), h
    bound, iters = engine.unbind_plain_f64(_groups(small), *X.T, *V.T, M, max_iter=max_iter)
    assert torch.equal(r.bound, bound)
    assert np.array_equal(r.iters.cpu().numpy(), iters)
