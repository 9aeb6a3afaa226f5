"""The softened sums at FP64 test points within their documented bounds of FP64 (S 2^-20, a and
w 2^-19 of the sum of |terms|): tests spread over a halo and others within an FP32 ulp of a
source's coordinates, where the lo part of the test decides the difference; few tests (lanes
over the sources) and many (tiles)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 5e-4


@pytest.mark.parametrize("tests", [8, 9, 200])
@pytest.mark.parametrize("n", [7, 1025, 20000])
def test_soft_sums_within_their_bounds(gpu, tests, n):
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(n + tests)
    x = (rng.normal(scale=0.004, size=(n, 3)) + [17.0, -9.0, 3.0]).astype(np.float32)
    m = np.exp(rng.uniform(np.log(1e4), np.log(1e6), n)).astype(np.float32)
    t = rng.normal(scale=0.004, size=(tests, 3)) + [17.0, -9.0, 3.0]
    near = x[rng.integers(0, n, tests // 2)].astype(np.float64)
    t[: tests // 2] = near + rng.uniform(-1, 1, near.shape) * np.spacing(np.abs(near).astype(np.float32))
    print(f"n={n} tests={tests}", flush=True)
    r = engine.pot_soft_batched(np.array([0, n]), m, *x.T, np.array([0, tests]), *t.T, EPS,
                                pot=True, acc=True, wsum=True)
    d = torch.from_numpy(x).cuda().double()[None] - torch.from_numpy(t).cuda()[:, None]
    keep = (d != 0).all(2)
    w = torch.rsqrt((d * d).sum(2) + EPS * EPS) * keep
    mm = torch.from_numpy(m).cuda().double()
    S, w3 = (mm * w).sum(1), mm * w ** 3
    a, mag = (w3[:, :, None] * d).sum(1), (w3[:, :, None] * d.abs()).sum(1)
    assert bool(((r["pot"] - S).abs() <= 2.0 ** -20 * S).all())
    assert bool(((r["acc"] - a).abs() <= 2.0 ** -19 * mag).all())
    assert bool(((r["wsum"] - w3.sum(1)).abs() <= 2.0 ** -19 * w3.sum(1)).all())


def test_kept_sources_stay_on_their_stream(gpu):
    """The packed sources that soft_potential keeps are ordered with the stream that packed
    them: another stream packs its own, the same one finds them."""
    import torch

    from pyhalma_amd import centring

    centring.clear_cache()
    pos, m = torch.rand(1000, 3, device="cuda"), torch.rand(1000, device="cuda")
    print("streams", flush=True)
    a = centring._src_packed(pos, m)
    assert centring._src_packed(pos, m) is a
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        b = centring._src_packed(pos, m)
        cols = centring._src_cols(pos)
        assert b is not a and centring._src_packed(pos, m) is b
    assert centring._src_cols(pos)[0] is not cols[0]
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    centring.clear_cache()
