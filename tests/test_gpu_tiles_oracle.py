"""Each P2G tile (pages by 512 or 256 threads, 2x2x2-page blocks by 512 or 256)
against the oracle on cells that hold from none to many particles: the clumped
scene as the first of a batch whose second scene, single particles here and
there, brings the block count into the tile's range.  The count, from the page
tables, is checked against the lines of the dispatch (in blocks: 30, 85 and 400 %
of 256 CUs, the last 200 % for APIC).  The bars are those of one substep."""
import numpy as np
import pytest

from conftest import max_rel_field, oracle_params
from test_gpu_tiles import clumps, params

pytestmark = pytest.mark.gpu
CU = 256
REF = {}


def reference(mpmx, oracle, transfer):
    if transfer not in REF:
        x, v = clumps(20000, 64, 7)
        m = np.full(len(x), 1e-4)
        sim = oracle.Sim(oracle_params(oracle, params(mpmx, 64, transfer)), x.astype(np.float32),
                         v.astype(np.float32), m.astype(np.float32))
        for _ in range(2):
            sim.substep(1e-4)
        REF[transfer] = x, v, {k: sim.get(k) for k in ("x", "v", "F", "B")}
    return REF[transfer]


@pytest.mark.parametrize("transfer", [0, 1])
@pytest.mark.parametrize("tile,filler", [("page 512", 5), ("page 256", 50), ("block 512", 150), ("block 256", 20000)])
def test_tile_against_oracle(mpmx, oracle, tile, filler, transfer):
    x, v, want = reference(mpmx, oracle, transfer)
    n = len(x)
    xf = np.random.default_rng(6).uniform(0.1, 0.9, (filler, 3)).astype(np.float32).astype(np.float64)
    ctx = mpmx.Context([params(mpmx, 64, transfer), params(mpmx, 128, transfer)])
    ctx.set_particles_batch([n, filler], np.concatenate([x, xf]), np.concatenate([v, np.zeros_like(xf)]),
                            np.full(n + filler, 1e-4))
    blocks = len(np.unique(ctx.tables()["page_key"] >> np.uint64(3)))
    lines = [0, 0.30 * CU, 0.85 * CU, (4 if transfer == 0 else 2) * CU, 1e9]
    k = ["page 512", "page 256", "block 512", "block 256"].index(tile)
    assert lines[k] < blocks <= lines[k + 1], blocks
    ctx.run(2, 1e-4)
    ctx.sync()
    for k, tol in (("x", 1e-6), ("v", 1e-4), ("F", 1e-5), ("B", 1e-3)):
        assert max_rel_field(ctx.get(k)[:n], want[k]) < tol, k
