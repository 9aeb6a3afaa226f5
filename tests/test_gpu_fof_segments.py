"""FoF labels of a dense core with long columns of cells in fields of cells below and above
2^19 in all, where columns are linked cell by cell and four cells at a time (equal to the
oracle's)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field", [3000, 400000, 700000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_fof_core_in_a_field(gpu, field, dtype):
    from pyhalma_amd import engine

    rng = np.random.default_rng(field)
    side = 3.0 * field ** (1 / 3)  # ll = 1: nearly every field particle has its own cell
    core = rng.normal(size=(20000, 3)) * [1.0, 1.0, 6.0] + side / 2
    ladder = np.stack([np.full(600, 5.0), np.full(600, 5.0), np.arange(600) * 0.58], 1)
    ladder[:, 2] %= side
    x = np.concatenate([rng.uniform(0, side, (field, 3)), core, ladder]).astype(dtype)
    x = np.ascontiguousarray(x[rng.permutation(len(x))])
    got = engine.fof_labels(*x.T, 1.0).cpu().numpy()
    assert np.array_equal(got, oracle.fof_labels_cells(*x.T, 1.0))
