"""The centring iteration on the device (halma_refine_centres) against the same iteration
in FP64 torch: haloes of sizes around its 2048-particle chunks and its 512-particle inner
step, empty and one-particle haloes, iteration limits around its batches of four,
limits below 0 and beyond any count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 5e-4


def _fp64(x, m, c, tol, max_iter):
    """(centre, S, steps taken, last step) of one halo, x (n, 3) float64."""
    it, length = 0, float("inf")
    for _ in range(max_iter):
        d = x - c
        w = m * ((d * d).sum(1) + EPS * EPS) ** -1.5
        w = np.where((d != 0).all(1), w, 0.0)
        step = (w[:, None] * d).sum(0) / w.sum() if w.sum() > 0 else np.zeros(3)
        c = c + step
        it, length = it + 1, float(np.sqrt((step ** 2).sum()))
        if not length > tol * EPS:
            break
    d = x - c
    s = np.where((d != 0).all(1), m * ((d * d).sum(1) + EPS * EPS) ** -0.5, 0.0)
    return c, s.sum(), it, length


@pytest.mark.parametrize("max_iter", [0, 1, 4, 5, 9, 200])
def test_refine_centres_chunk_edges(gpu, max_iter):
    from pyhalma_amd import centring

    rng = np.random.default_rng(3)
    sizes = [0, 1, 511, 513, 2047, 2048, 2049, 0, 4097, 10000]
    off = np.concatenate([[0], np.cumsum(sizes)])
    n, H = int(off[-1]), len(sizes)
    x = np.empty((n, 3), np.float32)
    seeds = np.zeros((H, 3))
    for h in range(H):
        cen = rng.uniform(-20, 20, 3)
        u = np.sqrt(rng.uniform(1e-6, 0.99, sizes[h]))
        v = rng.normal(size=(sizes[h], 3))
        v /= np.maximum(np.linalg.norm(v, axis=1, keepdims=True), 1e-30)
        x[off[h]:off[h + 1]] = cen + (0.004 * u / (1 - u))[:, None] * v
        seeds[h] = cen + rng.normal(scale=5e-4, size=3)
    m = rng.uniform(1e4, 1e6, n).astype(np.float32)
    print(f"max_iter={max_iter} n={n}", flush=True)
    r = centring.refine_centres(*x.T, m, off, seeds, EPS, max_iter=max_iter, tol=1e-3)
    c, S = r.centres.cpu().numpy(), r.S.cpu().numpy()
    iters, steps = r.iters.cpu().numpy(), r.steps.cpu().numpy()
    for h in range(H):
        sl = slice(off[h], off[h + 1])
        want, ws, it, length = _fp64(x[sl].astype(np.float64), m[sl].astype(np.float64),
                                     seeds[h].copy(), 1e-3, max_iter)
        # a step's error is the sums' 1e-6 of the halo's w-weighted extent (about EPS); the
        # iteration contracts, so its errors do not build up beyond a few of them
        assert np.linalg.norm(c[h] - want) <= 2e-5 * EPS, h
        if sizes[h] == 1:
            continue  # arrived on its only particle up to rounding: the rule's pair or none
        assert abs(S[h] - ws) <= 2e-6 * ws, h
        assert abs(int(iters[h]) - it) <= 1, h
        if iters[h] == it and np.isfinite(length):
            assert abs(steps[h] - length) <= 2e-5 * EPS, h
        elif it == 0:
            assert np.isinf(steps[h])


def test_refine_centres_any_limit(gpu):
    """Limits beyond any count (2^31 - 1 and 10^10 among them) are no limit, those below 0
    are 0, as a loop over range(max_iter) has it."""
    from pyhalma_amd import centring

    rng = np.random.default_rng(8)
    off = np.array([0, 700, 3000])
    x = rng.normal(scale=0.004, size=(3000, 3)).astype(np.float32)
    m = rng.uniform(1e4, 1e6, 3000).astype(np.float32)
    seeds = rng.normal(scale=1e-3, size=(2, 3))
    print("limits", flush=True)

    def run(max_iter):
        r = centring.refine_centres(*x.T, m, off, seeds, EPS, max_iter=max_iter, tol=1e-3)
        return [a.cpu().numpy() for a in (r.centres, r.S, r.iters, r.steps)]

    want, none = run(2000), run(0)
    assert 0 < want[2].max() < 2000 and none[2].max() == 0
    for max_iter in (2 ** 31 - 2, 2 ** 31 - 1, 2 ** 31, 10 ** 10):
        for a, b in zip(run(max_iter), want):
            assert np.array_equal(a, b), max_iter
    for a, b in zip(run(-1), none):
        assert np.array_equal(a, b)
