"""Page tiles and block tiles of the gathers: a scene of few blocks runs its
gathers by pages, inside a batch with many blocks by 2x2x2-page blocks, and both
must give the same bits; cells hold from none to many particles, odd and even
numbers of them, at every place of a tile."""
import numpy as np
import pytest

from conftest import max_rel_field, oracle_params

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "F", "B", "c", "alpha", "psi", "g")


def clumps(n, N, seed):
    """n particles in 13^3 cells around the middle, cell counts over two decades."""
    rng = np.random.default_rng(seed)
    w = 10.0 ** rng.uniform(-1.5, 1.0, 13 ** 3)
    cell = rng.choice(13 ** 3, size=n, p=w / w.sum())
    ijk = np.stack([cell // 169, (cell // 13) % 13, cell % 13], 1) + N // 2 - 6
    x = (ijk + rng.uniform(0.02, 0.98, (n, 3))) / N
    v = rng.normal(0.0, 0.3, (n, 3))
    return x.astype(np.float32).astype(np.float64), v.astype(np.float32).astype(np.float64)


def params(mpmx, N, transfer):
    return mpmx.default_params(N=N, transfer=transfer, E=1e4, nu=0.3, V0=1e-7, yield_stress=100.0,
                               gravity=(0.0, -9.8, 0.0))


@pytest.mark.parametrize("precision", ["fp32", "mixed", "mixed_f16"])
@pytest.mark.parametrize("transfer", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 1023, 20000])
def test_pages_equal_blocks(mpmx, n, transfer, precision):
    prec = {"fp32": mpmx.FP32, "mixed": mpmx.MIXED, "mixed_f16": mpmx.MIXED_F16}[precision]
    cfg = mpmx.default_config(precision=prec)
    x, v = clumps(n, 64, 5)
    m = np.full(n, 1e-4)
    rng = np.random.default_rng(6)
    nf = 20000   # one particle here and there in 102^3 cells: some 2,000 blocks
    xf = rng.uniform(0.1, 0.9, (nf, 3)).astype(np.float32).astype(np.float64)
    pa, pf = params(mpmx, 64, transfer), params(mpmx, 128, transfer)
    alone = mpmx.Context(pa, cfg)
    alone.set_particles(x, v, m)
    batch = mpmx.Context([pa, pf], cfg)
    batch.set_particles_batch([n, nf], np.concatenate([x, xf]), np.concatenate([v, np.zeros((nf, 3))]),
                              np.full(n + nf, 1e-4))
    for steps in (1, 4):
        for ctx in (alone, batch):
            ctx.run(steps, 1e-4)
            ctx.sync()
        for k in FIELDS:
            assert np.array_equal(alone.get(k), batch.get(k)[:n]), (steps, k)
    assert alone.stats()["numPage"] * 8 < batch.stats()["numPage"]


@pytest.mark.parametrize("transfer", [0, 1])
def test_clumped_substep_against_oracle(mpmx, oracle, transfer):
    """Two substeps (block tiles, then page tiles) at the one-substep bars."""
    x, v = clumps(20000, 64, 7)
    p = params(mpmx, 64, transfer)
    m = np.full(len(x), 1e-4)
    ctx = mpmx.Context(p)
    ctx.set_particles(x, v, m)
    sim = oracle.Sim(oracle_params(oracle, p), x.astype(np.float32), v.astype(np.float32), m.astype(np.float32))
    for _ in range(2):
        ctx.run(1, 1e-4)
        ctx.sync()
        sim.substep(1e-4)
    for k, tol in (("x", 1e-6), ("v", 1e-4), ("F", 1e-5), ("B", 1e-3)):
        assert max_rel_field(ctx.get(k), sim.get(k)) < tol, k
