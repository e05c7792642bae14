"""The one-workgroup sort of few movers: from no mover at all up to its capacity
(16,384) and past it (its tile-by-tile form in global memory), at particle
counts around its tiles, it gives the order of the radix sort of every key."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 2047, 2049, 16385, 64000])
@pytest.mark.parametrize("shift", [0.0, 0.002, 0.03, 0.24, 0.27, 0.6])
def test_few_movers_order(mpmx, n, shift):
    """A stress-free block at rest takes a substep (no mover is published, so
    the next sort foresees few), then flies `shift` cells per substep: about
    that share of its particles changes cell at once."""
    p, x, v, m, dt = mpmx.scene(0, seed=3, scale=1.0)
    p.gravity[:] = [0.0, 0.0, 0.0]
    x, v, m = x[:n], np.zeros_like(v[:n]), m[:n]
    dt = 1e-3
    speed = shift / p.N / dt
    ctxs = []
    for variant in (1, 2):
        ctx = mpmx.Context(p, mpmx.default_config(sort_variant=variant))
        ctx.set_particles(x, v, m)
        ctxs.append(ctx)
    for ctx in ctxs:
        ctx.run(2, dt)
    for rep in range(3):
        for ctx in ctxs:
            ctx.set("v", np.tile([speed, 0.6 * speed, -0.3 * speed], (n, 1)))
            ctx.set("B", np.zeros((n, 3, 3)))
            ctx.set("F", np.tile(np.eye(3), (n, 1, 1)))
            ctx.substep(dt)
            ctx.bin_sort()
        (oa, ka), (ob, kb) = ctxs[0].order(), ctxs[1].order()
        assert np.array_equal(ka, kb), rep
        assert np.array_equal(oa, ob), rep
    assert np.array_equal(ctxs[0].get("x"), ctxs[1].get("x"))
