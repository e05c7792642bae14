"""Captured substeps between other calls: what the replays leave on the host (which
tables and fields are current, which keys are sorted) is what the eager launches
leave, so that every later call gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "F", "B", "c", "alpha", "psi", "g")


def pair(mpmx, **cfg):
    out = []
    for graph in (1, 0):
        p, x, v, m, dt = mpmx.scene(3, seed=1, scale=0.1)
        ctx = mpmx.Context(p, mpmx.default_config(use_graph=graph, **cfg))
        ctx.set_particles(x, v * 2.0, m)
        out.append(ctx)
    return out, dt


def same(g, e, tag):
    og, kg = g.order()
    oe, ke = e.order()
    assert np.array_equal(og, oe) and np.array_equal(kg, ke), tag
    for k in FIELDS:
        assert np.array_equal(g.get(k), e.get(k)), (tag, k)


@pytest.mark.parametrize("variant", [1, 2])
def test_tables_after_replays(mpmx, variant):
    """The page and virtual-page tables, read between the replays."""
    (g, e), dt = pair(mpmx, p2g_variant=variant)
    for rep in range(4):
        for ctx in (g, e):
            ctx.run(5, dt)
        tg, te = g.tables(), e.tables()
        for k in te:
            assert np.array_equal(tg[k], te[k]), (rep, k)


def test_stress_fields_after_replays(mpmx):
    """A replay does not store sigma; the field of an older stress pass is refused."""
    (g, e), dt = pair(mpmx)
    for ctx in (g, e):
        ctx.run(6, dt)
        ctx.bin_sort()
        ctx.rebuild()
        ctx.stress()
        ctx.get("sigma")
        ctx.run(6, dt)
        with pytest.raises(mpmx.MpmxError) as err:
            ctx.get("sigma")
        assert err.value.status == mpmx.ERR_ARG
    same(g, e, "after")


@pytest.mark.parametrize("sort_variant", [0, 1, 2])
def test_replays_after_a_sort_without_tables(mpmx, sort_variant):
    """Stage calls that sort and move the particles without building the tables: the
    next movers' places do not come from those tables, in a replay either."""
    (g, e), dt = pair(mpmx, sort_variant=sort_variant)
    for rep in range(3):
        for ctx in (g, e):
            ctx.run(5, dt)
            ctx.bin_sort()
            ctx.g2p(dt)
            ctx.run(4, dt)
        same(g, e, rep)
