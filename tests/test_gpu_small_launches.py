"""Pair sums of launches too small for the tuned source chunk, on the GPU: within the
library's error bound of the FP64 sum at the edges of the chunks and test tiles."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 127, 129, 511, 513, 3001, 8191])
@pytest.mark.parametrize("nt", [1, 127, 129, 797, 2049])
def test_small_launches(gpu, ns, nt):
    from pyhalma_amd import engine

    rng = np.random.default_rng(ns * 3000 + nt)
    x, y, z = (rng.normal(size=ns + nt).astype(np.float32) for _ in range(3))
    m = rng.uniform(0.5, 2.0, ns).astype(np.float32)
    s, t = slice(0, ns), slice(ns, None)
    got = engine.pot_sum(m, x[s], y[s], z[s], x[t], y[t], z[t], out_dtype=np.float64).cpu().numpy()
    want = oracle.pot_sum_f64(m, x[s], y[s], z[s], x[t], y[t], z[t])
    assert (np.abs(got - want) <= engine.pot_error_bound() * want).all()
