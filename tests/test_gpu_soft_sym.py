"""The symmetric softened self sums (S and a of every member over its halo, no wsum) against
FP64: halo sizes at the edges of the 8-source groups, the 128- and 512-member blocks, the
64-block bands and the size from which blocks hold 512 members; equal coordinates and
duplicates; each output alone; a halo's bits independent of the other haloes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 5e-4
U = 2.0 ** -24


def _fp64(p, i):
    """(S, a, sum of |terms| of a) of rows i against all rows p (n, 4) in float64."""
    import torch

    d = p[None, :, :3] - p[i, None, :3]
    w = torch.rsqrt((d * d).sum(2) + EPS * EPS) * (d != 0).all(2)
    t = (p[:, 3] * w ** 3)[:, :, None] * d
    return (p[:, 3] * w).sum(1), t.sum(1), t.abs().sum(1)


def _halo(rng, n, dup):
    x = rng.normal(scale=0.004, size=(n, 3)) * rng.uniform(0.05, 1, (n, 1)) + rng.uniform(-20, 20, 3)
    x = x.astype(np.float32)
    if dup and n > 4:
        x[n // 2] = x[0]                       # a duplicate
        x[n // 3, 1] = x[n - 1, 1]             # one equal coordinate
    m = rng.uniform(1e4, 1e6, n).astype(np.float32)
    return np.concatenate([x, m[:, None]], 1)


@pytest.mark.parametrize("sizes", [
    [1, 0, 2, 7, 8, 9, 65], [127, 128, 129], [511, 512, 513, 1000], [8191, 8193, 16383],
    [16384, 16385], [32768, 32769], [66000, 300]])
def test_self_sums_block_and_band_edges(gpu, sizes):
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(sum(sizes))
    rows = torch.from_numpy(np.concatenate([_halo(rng, n, True) for n in sizes])).cuda()
    off = np.concatenate([[0], np.cumsum(sizes)])
    print(f"sizes={sizes}", flush=True)
    r = engine.pot_soft_self(off, rows, EPS, pot=True, acc=True)
    S, a = r["pot"], r["acc"]
    for h, n in enumerate(sizes):
        if n == 0:
            continue
        p = rows[off[h]:off[h + 1]].double()
        i = torch.from_numpy(np.unique(np.concatenate([
            np.arange(min(n, 520)), np.arange(max(0, n - 520), n), rng.integers(0, n, 200)]))).cuda()
        step = max(1, 20_000_000 // n)
        for k in range(0, i.numel(), step):
            q = i[k:k + step]
            ws, wa, mag = _fp64(p, q)
            # per term: differences and r^2 2.5u, the root 2u, the product and eight terms in
            # FP32 8u, 0.5u for the FP64 sums (S); three times the root's error, two products,
            # the difference and the sums for a
            es = (S[off[h] + q] - ws).abs() / ws.clamp(min=1e-300)
            assert float(es.max()) <= 13 * U or n == 1, (h, float(es.max()))
            ea = (a[off[h] + q] - wa).abs() / mag.clamp(min=1e-300)
            assert float(ea.max()) <= 26 * U or n == 1, (h, float(ea.max()))
    one = engine.pot_soft_self(off, rows, EPS, pot=True, acc=False)["pot"]
    two = engine.pot_soft_self(off, rows, EPS, pot=False, acc=True)["acc"]
    assert torch.equal(one, S) and torch.equal(two, a)
    h = len(sizes) - 1                                       # the last halo on its own
    alone = engine.pot_soft_self(off[h:] - off[h], rows[off[h]:], EPS, pot=True, acc=True)
    assert torch.equal(alone["pot"], S[off[h]:]) and torch.equal(alone["acc"], a[off[h]:])
    based = engine.pot_soft_self(off[h:], rows, EPS, pot=True, acc=True)  # offsets not from 0
    assert torch.equal(based["pot"][off[h]:], S[off[h]:])
    # the sums with wsum run one-sided: the same values to both bounds (13u and 15u)
    old = engine.pot_soft_self(off, rows, EPS, pot=True, acc=True, wsum=True)
    assert float(((old["pot"] - S).abs() / S.clamp(min=1e-300)).max()) <= 28 * U


@pytest.mark.parametrize("n", [1000, 16383, 17000])
def test_self_sums_are_as_exact_as_the_one_sided_ones(gpu, n):
    """Both forms add eight terms in FP32 before FP64 (or a Kahan pair), on either side of a
    pair: the spread of S about its FP64 value is no larger (the mean, the root's bias, is
    common to both).  With 64 terms in FP32 on the source side it is 1.36 of it at 17000."""
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(n)
    u = np.sqrt(rng.uniform(1e-6, 0.98, n))
    v = rng.normal(size=(n, 3))
    x = (0.02 * u / (1 - u))[:, None] * v / np.linalg.norm(v, axis=1, keepdims=True)
    m = np.exp(rng.uniform(np.log(1e4), np.log(1e6), n))
    rows = torch.from_numpy(np.concatenate([x + 7, m[:, None]], 1).astype(np.float32)).cuda()
    print(f"n={n}", flush=True)
    off, p = np.array([0, n]), rows.double()
    S = engine.pot_soft_self(off, rows, EPS, pot=True)["pot"]
    T = engine.pot_soft_self(off, rows, EPS, pot=True, wsum=True)["pot"]
    want = torch.cat([_fp64(p, torch.arange(k, min(k + 500, n), device="cuda"))[0]
                      for k in range(0, n, 500)])
    sym, one = ((S - want) / want).std(), ((T - want) / want).std()
    print(f"symmetric {float(sym):.3e} one-sided {float(one):.3e}", flush=True)
    assert float(sym) <= 1.05 * float(one)


@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 1])
def test_self_sums_large_haloes_by_their_own_size(gpu, n):
    """Above 2^21 members a halo is one-sided; a small halo of the same call keeps its bits
    either way, and the large one is within the bound."""
    import torch

    from pyhalma_amd import engine

    rng = np.random.default_rng(n)
    rows = torch.from_numpy(np.concatenate([_halo(rng, n, True), _halo(rng, 700, True)])).cuda()
    off = np.array([0, n, n + 700])
    print(f"n={n}", flush=True)
    r = engine.pot_soft_self(off, rows, EPS, pot=True, acc=True)
    p = rows[:n].double()
    i = torch.from_numpy(np.concatenate([np.arange(9), rng.integers(0, n, 40),
                                         np.arange(n - 9, n)])).cuda()
    for q in i.split(16):
        ws, wa, mag = _fp64(p, q)
        assert float(((r["pot"][q] - ws).abs() / ws).max()) <= 15 * U
        assert float(((r["acc"][q] - wa).abs() / mag).max()) <= 28 * U
    alone = engine.pot_soft_self(off[1:] - n, rows[n:], EPS, pot=True, acc=True)
    assert torch.equal(alone["pot"], r["pot"][n:]) and torch.equal(alone["acc"], r["acc"][n:])
    one = engine.pot_soft_self(off[:2], rows, EPS, pot=True, acc=True, wsum=True)
    assert torch.equal(one["pot"], r["pot"][:n]) == (n > 1 << 21)
