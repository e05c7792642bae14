"""The FP64 stress update from the principal axes (columns of F V made orthogonal)
where it can go wrong: reflections, singular values far apart (both sides of the
ratio 1e-5 below which the smallest direction is completed from the others), a
singular value of zero, nearly equal ones, and none to turn (diagonal F).

Bound: outputs are FP64 results rounded to FP32 (6e-8); the oracle's QR iteration
stops at 128 eps = 3e-14 of the largest singular value, 3e-8 of the smallest at the
ratio 1e-6 used here, which enters the flow through its logarithm (of order 10).
1e-6 of each particle's largest entry, the bar of the other stress tests."""
import numpy as np
import pytest

from conftest import oracle_params

pytestmark = pytest.mark.gpu


def rotations(rng, n):
    q = rng.standard_normal((n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)


def gradients(kind, n, rng):
    s = rng.uniform(0.6, 1.8, (n, 3))
    s += 0.05 * np.arange(3)   # no two equal
    if kind == "reflected":
        s[:, 2] = -rng.uniform(0.1, 0.5, n)
    elif kind == "thin":
        s[:, 2] = 10.0 ** rng.uniform(-6.0, -1.0, n)
    elif kind == "thin_reflected":
        s[:, 2] = -(10.0 ** rng.uniform(-6.0, -1.0, n))
    elif kind == "close":
        s[:, 1] = s[:, 0] * (1 + 10.0 ** rng.uniform(-4.0, -2.0, n))
    elif kind == "flat":
        s[:, 2] = 0.0
    S = np.zeros((n, 3, 3))
    for k in range(3):
        S[:, k, k] = s[:, rng.permutation(3)[k] if kind == "diagonal" else k]
    if kind in ("diagonal", "flat"):
        return S
    return rotations(rng, n) @ S @ rotations(rng, n)


@pytest.mark.parametrize("kind", ["ordinary", "reflected", "thin", "thin_reflected", "close", "diagonal", "flat"])
def test_principal_axes(mpmx, oracle, kind):
    p, x, v, m, dt = mpmx.scene(0, seed=1, scale=0.25)
    ctx = mpmx.Context(p)
    ctx.set_particles(x, v, m)
    n = ctx.n
    rng = np.random.default_rng(11)
    ins = {"F": gradients(kind, n, rng), "c": rng.uniform(0.3, 1.0, n), "g": rng.uniform(0.1, 1.0, n),
           "alpha": rng.uniform(0.0, 0.9, n), "psi": np.zeros(n)}
    ins = {k: a.astype(np.float32).astype(np.float64) for k, a in ins.items()}
    op = oracle_params(oracle, p)
    ref = [oracle.von_mises(op, ins["F"][i], ins["c"][i], ins["g"][i], ins["alpha"][i], 0.0) for i in range(n)]
    # a state without flow keeps J = 0, for which the energy has no value
    use = np.array([np.all(np.isfinite(r["sigma"])) for r in ref])
    assert use.mean() > 0.2
    ins["F"][~use] = np.eye(3)
    for k, a in ins.items():
        ctx.set(k, a)
    ctx.stress()
    # (V is V0 times the determinant of F; the constants' FP32 rounding times a log
    # strain of 14 moves it more than the bound, F and sigma less)
    for k in ("F", "sigma", "FP", "alpha", "psi"):
        got = ctx.get(k).reshape(n, -1)[use]
        want = np.array([np.ravel(r[k]) for r in ref])[use]
        scale = np.abs(want).max(axis=1, keepdims=True) + 1e-30
        if k in ("alpha", "psi"):
            scale = np.maximum(scale, 1.0)
        err = np.abs(got - want) / scale
        assert err.max() < 1e-6, (k, err.max())
