"""FoF labels where links cross the stretches of consecutive cells that a workgroup joins by
itself: cell counts around the stretch sizes (256 and up, 2048 from 2.1M cells on), chains
along each axis, lattices with spacings below, at and above the linking length, uniform
boxes that percolate (every component spans many stretches), equal to the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _check(x, ll):
    from pyhalma_amd import engine

    x = np.ascontiguousarray(x)
    print(f"n={len(x)} ll={ll} {x.dtype}", flush=True)
    got = engine.fof_labels(*x.T, ll).cpu().numpy()
    assert np.array_equal(got, oracle.fof_labels_c(*x.T, ll))


@pytest.mark.parametrize("n", [255, 256, 257, 511, 513, 1023, 4097])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_fof_chains(gpu, n, axis):
    rng = np.random.default_rng(n)
    x = rng.uniform(0, 0.3, (n, 3))
    x[:, axis] = np.arange(n) * 0.9 + rng.uniform(-0.04, 0.04, n)   # one cell each or two
    x[n // 2:, axis] += 3.0                                          # one gap
    _check(x[rng.permutation(n)], 1.0)


@pytest.mark.parametrize("spacing", [0.55, 1.0, 1.01])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_fof_lattices(gpu, spacing, dtype):
    g = np.stack(np.meshgrid(*[np.arange(k) for k in (23, 17, 29)], indexing="ij"), -1)
    x = (g.reshape(-1, 3) * spacing).astype(dtype)
    _check(x[np.random.default_rng(2).permutation(len(x))], 1.0)


@pytest.mark.parametrize("n,mean", [(40000, 1.3), (40000, 0.9), (300000, 0.95), (2600000, 1.05)])
def test_fof_uniform_boxes(gpu, n, mean):
    # ll = 1, mean spacing `mean`: 0.86 percolates
    rng = np.random.default_rng(n)
    _check(rng.uniform(0, mean * n ** (1 / 3), (n, 3)).astype(np.float32), 1.0)


@pytest.mark.parametrize("side", [8, 15, 16, 17, 23])
@pytest.mark.parametrize("spacing", [0.6, 0.99, 1.02])
def test_fof_slabs_about_a_stretch(gpu, side, spacing):
    """Slabs of one x of side^2 cells, shorter and longer than a stretch (256 cells), so that
    some stretches hold neighbours in x and others only own columns and neighbours in y; full
    slabs beside sparse and empty ones."""
    rng = np.random.default_rng(side)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 2, indexing="ij"), -1).reshape(-1, 2)
    parts = []
    for k in range(40):
        yz = g if k % 7 < 4 else g[rng.permutation(len(g))[: (0, 9, len(g) // 2)[k % 3]]]
        parts.append(np.concatenate([np.full((len(yz), 1), k), yz], 1))
    x = np.concatenate(parts) * spacing
    _check(x[rng.permutation(len(x))], 1.0)


@pytest.mark.parametrize("n", [255, 256, 257, 258, 5000, 70001])
def test_fof_long_columns(gpu, n):
    """Columns of about 256 cells and far beyond along z (spread over a wavefront when they are
    listed), beside short ones, with gaps and side links."""
    rng = np.random.default_rng(n)
    z = np.arange(n) * 0.58 + rng.uniform(0, 1e-3, n)
    z[n // 3:] += 2.0
    a = np.stack([np.zeros(n), np.zeros(n), z], 1) + rng.uniform(0, 1e-3, (n, 3))
    b = np.stack([np.full(n, 1.1), np.full(n, 0.7), z[::-1]], 1)[:: 7]
    c = rng.uniform(0, 3, (500, 3)) + [0, 0, 0.58 * n / 2]
    x = np.concatenate([a, b, c])
    _check(x[rng.permutation(len(x))], 1.0)
