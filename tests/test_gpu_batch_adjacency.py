"""The page adjacency of a batch whose scenes fill their slots of the page space to
the last page (the grid is a power of two): the neighbour past a scene's domain
is none, whichever scene or none has the slot its key falls into."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def unmorton(k):
    xyz = [0, 0, 0]
    for b in range(10):
        for a in range(3):   # x at bit 2, y at 1, z at 0
            xyz[a] |= ((k >> (3 * b + 2 - a)) & 1) << b
    return xyz


def morton(x, y, z):
    k = 0
    for b in range(10):
        k |= ((z >> b) & 1) << (3 * b) | ((y >> b) & 1) << (3 * b + 1) | ((x >> b) & 1) << (3 * b + 2)
    return k


@pytest.mark.parametrize("scenes,N", [(2, 16), (5, 32), (17, 32)])
def test_neighbours_stay_in_their_scene(mpmx, scenes, N):
    rng = np.random.default_rng(3)
    n = 400
    # every scene reaches the first and the last page of each axis
    x = rng.uniform(2.2 / N, 1 - 2.2 / N, (scenes, n, 3))
    x[:, :8] = np.array([[a, b, c] for a in (2.2, N - 2.2) for b in (2.2, N - 2.2) for c in (2.2, N - 2.2)]) / N
    x = x.reshape(-1, 3).astype(np.float32).astype(np.float64)
    p = mpmx.default_params(N=N, E=1e4, nu=0.3, V0=1e-7, gravity=(0.0, 0.0, 0.0))
    ctx = mpmx.Context([p] * scenes)
    ctx.set_particles_batch([n] * scenes, x, np.zeros_like(x), np.full(scenes * n, 1e-4))
    t = ctx.tables()
    keys = t["page_key"].astype(np.int64)
    rank = {int(k): i for i, k in enumerate(keys)}
    shift = 3 * int(np.log2(N // 4))
    none = 0
    for page in range(t["numPage"]):
        k = int(keys[page])
        px, py, pz = unmorton(k)
        for q in range(7):
            o = q + 1
            nk = morton(px + (o >> 2 & 1), py + (o >> 1 & 1), pz + (o & 1))
            want = rank.get(nk, -1) if nk >> shift == k >> shift else -1
            none += want < 0
            assert t["adj"][q, page] == want, (page, q)
    assert none > 0
