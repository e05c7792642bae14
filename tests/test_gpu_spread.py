"""A body that spreads over many times its pages inside one call, without a solve
(no substep then waits for the counts): the launches follow the block count.  The
same substeps right after a call that reads the counts are the measure; launches
by the count of the first substep take 1.5 to 1.6 times as long."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DT = 1e-3


@pytest.mark.parametrize("edge", [20, 40])
def test_launches_follow_the_block_count(mpmx, edge):
    N = 256
    rng = np.random.default_rng(1)
    g = np.stack(np.meshgrid(*[np.arange(2 * edge)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = (N // 2 - edge // 2 + (g + 0.5) * 0.5 + rng.uniform(-0.24, 0.24, g.shape)) / N
    p = mpmx.default_params(N=N, model=0, E=1e-3, nu=0.3, V0=0.125 / N ** 3, gravity=(0.0, 0.0, 0.0))
    best = []
    for _ in range(2):
        ctx = mpmx.Context(p, mpmx.default_config(max_pages=60000))
        ctx.set_particles(x.astype(np.float32).astype(np.float64), (x - 0.5) * 0.008 / DT,
                          np.full(len(x), 125.0 / N ** 3))
        ctx.run(150, DT)
        old = ctx.time_run(40, DT)   # reads the counts at its end
        best.append(old / ctx.time_run(40, DT))
        ctx.close()
    assert min(best) < 1.25, best
