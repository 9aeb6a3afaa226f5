"""The symmetric pair kernel's two launch forms (a wavefront per block pair from 4096 pairs
on, a workgroup of sixteen below) give the same bits, on coordinates rounded so that equal
ones are common (the rule's pair-by-pair branch), and within the bound of FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [0.0, 2e-6, 2e-4])
def test_pot_sym_wave_and_workgroup_forms(gpu, grid):
    import torch

    from pyhalma_amd import engine, synth

    rng = np.random.default_rng(31)
    # 196 haloes of 21 block pairs and edges of strips, segments and blocks: 4.2k pairs
    sizes = np.array([3000] * 196 + [1, 31, 33, 64, 65, 480, 511, 513, 1025])
    off = np.concatenate([[0], np.cumsum(sizes)])
    P = np.concatenate([synth.plummer_positions(rng, n, 0.005) + rng.uniform(-20, 20, 3)
                        for n in sizes])
    P = (np.round(P / grid) * grid if grid else P).astype(np.float32)
    m = rng.uniform(1e4, 1e6, len(P)).astype(np.float32)
    print(f"grid={grid} n={len(P)}", flush=True)
    got = engine.pot_sum_self(off, m, *P.T)
    for h in [0, 97, 195] + list(range(196, len(sizes))):
        s = slice(int(off[h]), int(off[h + 1]))
        alone = engine.pot_sum_self([0, sizes[h]], m[s], *P[s].T)
        assert torch.equal(alone, got[s]), h
        x = torch.from_numpy(P[s]).double().cuda()
        d = x[None] - x[:, None]
        w = torch.where((d != 0).all(2), torch.rsqrt((d * d).sum(2)), 0.0)
        want = (w * torch.from_numpy(m[s]).double().cuda()).sum(1)
        err = ((got[s] - want).abs() / want.clamp(min=1e-300)).max()
        assert float(err) <= engine.pot_sym_error_bound() or sizes[h] == 1, h
