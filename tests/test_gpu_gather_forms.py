"""Sphere queries and gas cells at the edges of their workgroup widths and sorts, on the GPU:
the sets, their order and the gas values are exact."""
import numpy as np
import pytest

from test_gpu_gathering import _amr_snapshot

pytestmark = pytest.mark.gpu


def _balls(counts, dtype, seed):
    # centre h holds counts[h] points within 0.3 of it; the centres are 1 apart
    rng = np.random.default_rng(seed)
    c = np.stack([np.arange(len(counts)) % 40, np.arange(len(counts)) // 40,
                  np.zeros(len(counts))], 1).astype(np.float64)
    own = np.repeat(np.arange(len(counts)), counts)
    d = rng.normal(size=(len(own), 3))
    d *= (rng.uniform(0, 0.29, len(own)) / np.linalg.norm(d, axis=1))[:, None]
    p = np.concatenate([c[own] + d, rng.uniform(3, 4, (500, 3)) + [0, 0, 2]])
    own = np.concatenate([own, np.full(500, -1)])
    order = rng.permutation(len(p))
    return c, p[order].astype(dtype), own[order]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("counts", [
    [1, 2, 3, 0, 255, 256, 257, 511, 513],            # one workgroup width of the sort
    [2047, 2048, 2049, 0, 1, 4096, 4097],             # both
    [16383, 16384, 5, 2048],                          # up to the largest sorted in LDS
    [16385, 70, 0, 2000],                             # one more: the radix passes
    [3] * 512,                                        # 16 wavefronts a centre on 256 CUs
    [2, 0, 4] * 171,                                  # four
])
def test_sphere_forms(gpu, counts, dtype):
    from pyhalma_amd import engine

    c, p, own = _balls(counts, dtype, len(counts))
    m = np.random.default_rng(2).uniform(0.5, 2, len(p))
    r = np.full(len(counts), 0.3)
    off, idx, sums = engine.ball_query(p[:, 0], p[:, 1], p[:, 2], c, r, m=m)
    _, loose, _ = engine.ball_query(p[:, 0], p[:, 1], p[:, 2], c, r, sorted=False)
    idx, loose = idx.cpu().numpy(), loose.cpu().numpy()
    assert np.diff(off).tolist() == list(counts)
    for h in range(len(counts)):
        want = np.nonzero(own == h)[0]
        assert np.array_equal(idx[off[h]:off[h + 1]], want)
        assert np.array_equal(np.sort(loose[off[h]:off[h + 1]]), want)
        np.testing.assert_allclose(sums[h], m[want].sum(), rtol=1e-13)


@pytest.mark.parametrize("sphere", [True, False])
def test_gas_cells_of_many_haloes(gpu, sphere):
    import torch

    from pyhalma_amd import gathering

    L, nc, levels, rx, ry, rz, cells = _amr_snapshot(4)
    grid = gathering.AmrGrid(L, nc, levels, *([c.shape[d] for c in cells[0]] for d in range(3)),
                             rx, ry, rz, cells)
    rng = np.random.default_rng(5)
    Q = 3000  # four wavefronts a halo, 16 for the parts below
    c = rng.uniform(-4, 4, (Q, 3))
    r = rng.uniform(0, 1.5, Q)
    box = np.stack([c[:, 0] - r, c[:, 0] + r, c[:, 1] - r, c[:, 1] + r, c[:, 2] - r,
                    c[:, 2] + r], 1)

    def run(a, b):
        return gathering.amr_particles(grid, 2.0, box[a:b], *((c[a:b], r[a:b]) if sphere else ()))

    off, gas = run(0, Q)
    assert off[-1] > 0
    for a in range(0, Q, 500):
        po, pg = run(a, a + 500)
        assert np.array_equal(po, off[a:a + 501] - off[a])
        for k in gas:
            assert torch.equal(pg[k], gas[k][off[a]:off[a + 500]])
