"""The P2G's tiles, pages by 512 or 256 threads and 2x2x2 blocks by 512 or 256, by
the number of blocks (the K s gather's pages alike): scenes alone on either side of
each line, and inside a batch of many blocks, by blocks of 256 threads.
The fixed-point sums do not depend on the tiling, so all must agree bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "F", "B", "c", "alpha", "psi", "g")


@pytest.mark.parametrize("precision", ["fp32", "mixed"])
@pytest.mark.parametrize("transfer", [0, 1])
@pytest.mark.parametrize("cells,n", [(20, 20001), (28, 30000), (46, 30000), (54, 40000), (75, 60000)])
# about 27, 64, 216, 340 and 1,000 blocks
def test_page_tiles_equal_blocks(mpmx, cells, n, transfer, precision):
    cfg = mpmx.default_config(precision=mpmx.FP32 if precision == "fp32" else mpmx.MIXED)
    N = 96 if cells > 50 else 64
    p = mpmx.default_params(N=N, transfer=transfer, E=1e4, nu=0.3, V0=1e-7, yield_stress=100.0)
    rng = np.random.default_rng(3)
    x = ((8 + rng.uniform(0.0, cells, (n, 3))) / N).astype(np.float32).astype(np.float64)
    v = rng.normal(0.0, 0.3, (n, 3)).astype(np.float32).astype(np.float64)
    pf = mpmx.default_params(N=128, transfer=transfer, E=1e4, nu=0.3, V0=1e-7, yield_stress=100.0)
    xf = rng.uniform(0.1, 0.9, (20000, 3)).astype(np.float32).astype(np.float64)
    alone = mpmx.Context(p, cfg)
    alone.set_particles(x, v, np.full(n, 1e-4))
    batch = mpmx.Context([p, pf], cfg)
    batch.set_particles_batch([n, 20000], np.concatenate([x, xf]), np.concatenate([v, np.zeros((20000, 3))]),
                              np.full(n + 20000, 1e-4))
    for ctx in (alone, batch):
        ctx.run(4, 1e-4)
        ctx.sync()
    for k in FIELDS:
        assert np.array_equal(alone.get(k), batch.get(k)[:n]), k
