"""Particles of infinite velocity in one cell: each adds the largest fixed-point
value to its nodes, and those of two must not cancel, so that the state is still
reported.  Every index that depends on a position is clamped to the grid."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def particles(mpmx, transfer, n):
    p = mpmx.default_params(N=64, transfer=transfer, E=1e4, nu=0.3, V0=1e-7, gravity=(0.0, 0.0, 0.0))
    rng = np.random.default_rng(2)
    x = ((30.0 + rng.uniform(0.6, 0.9, (n, 3))) / 64).astype(np.float32).astype(np.float64)
    ctx = mpmx.Context(p)
    ctx.set_particles(x, np.zeros_like(x), np.full(n, 1.0))
    ctx.set("v", np.full((n, 3), np.inf))
    return ctx


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_infinite_velocity_leaves_the_domain(mpmx, n):
    """APIC, no speed clamp: unit masses at some 1e9 cells per second."""
    ctx = particles(mpmx, 1, n)
    with pytest.raises(mpmx.MpmxError):
        ctx.run(1, 1e-4)
        ctx.sync()


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_infinite_velocity_on_the_grid(mpmx, n):
    """MLS: the nodes' momentum, 2^31 - 1 at least for every node of the cell."""
    ctx = particles(mpmx, 0, n)
    ctx.enable_p2g_copy()
    ctx.run(1, 1e-4)
    for ch in (1, 2, 3):
        g = ctx.grid(ch, p2g=True)
        assert np.count_nonzero(g) == 27 and g[g != 0].min() >= 2147483520.0, ch
