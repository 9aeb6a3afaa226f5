"""Per-halo masses and weighted sums at the edges of their chunks, on the GPU.

Double-double sums rounded once: within one unit of the last place (2^-52 relative) of the
exactly rounded sum of the same FP64 terms (math.fsum), sizes around the wavefront (64), the
unrolled step (256), the chunk (2048) and a halo of more than 64 chunks."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 63, 64, 65, 255, 257, 2047, 2048, 2049, 0, 4097, 64 * 2048 + 3]


@pytest.mark.parametrize("mt,tt", [(np.float32, np.float64), (np.float64, np.float32)])
@pytest.mark.parametrize("first", [0, 5])
def test_sums_at_the_chunk_edges(gpu, mt, tt, first):
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(4)
    off = first + np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int64)
    n = int(off[-1])
    m = 10.0 ** rng.uniform(-3, 3, n)
    m = m.astype(mt)
    t = (10.0 ** rng.uniform(3, 6, n)).astype(tt)
    t[::97] = 5e4  # not cold
    t[::101] = np.nan  # not cold
    bound = rng.integers(0, 2, n).astype(np.uint8)
    s = 10.0 ** rng.uniform(-8, 2, n)
    got = engine.gas_masses(off, torch.from_numpy(m).cuda(), torch.from_numpy(t).cuda(),
                            torch.from_numpy(bound).cuda()).cpu().numpy()
    w = engine.weighted_sums(off, torch.from_numpy(m).cuda(),
                             torch.from_numpy(s).cuda()).cpu().numpy()
    m64 = m.astype(np.float64)
    cold, b = t < 5e4, bound != 0
    ms = m64 * s
    for h in range(len(SIZES)):
        i = slice(off[h], off[h + 1])

        def total(keep):
            return math.fsum(m64[i][keep[i]])

        tot, cb = total(np.ones(n, bool)), total(cold & b)
        want = [tot, cb / tot if tot else 0.0, total(cold & ~b), total(~cold & ~b)]
        # the fraction is the rounded quotient of two such sums: three units
        np.testing.assert_allclose(got[h], want, rtol=3 * 2 ** -52, atol=0)
        np.testing.assert_allclose(w[h], math.fsum(ms[i]), rtol=2 ** -52, atol=0)


def test_no_haloes(gpu):
    import torch

    from pyhalma_amd import engine

    z = torch.zeros(0, dtype=torch.float64, device="cuda")
    b = torch.zeros(0, dtype=torch.uint8, device="cuda")
    assert engine.gas_masses([0], z, z, b).shape == (0, 4)
    assert engine.weighted_sums([0], z, z).shape == (0,)
    assert not engine.gas_masses([0, 0], z, z, b).cpu().numpy().any()
