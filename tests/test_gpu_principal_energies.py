"""The principal axes of the FP64 stress update under all three energies, the volume
of the final F, and gradients of exactly lower rank.

Bounds.  Outputs are FP64 results rounded to FP32, compared at 1e-6 of each
particle's largest entry, the bar of the other stress tests.  The device holds the
constants in FP32 (6e-8 of their value), and three of them multiply the log
strains in the exponents: 1.8e-7 of the largest |log strain|.  The oracle's QR
iteration stops at 128 eps = 3e-14 of the largest singular value: 3e-14 over the
ratio of the smallest to the largest."""
import numpy as np
import pytest

from conftest import oracle_params
from test_gpu_principal import gradients, rotations

pytestmark = pytest.mark.gpu
KINDS = ["ordinary", "reflected", "thin", "thin_reflected", "close", "diagonal"]


def setup(mpmx, model):
    p, x, v, m, dt = mpmx.scene(0, seed=1, scale=0.25)
    p.model = model
    ctx = mpmx.Context(p)
    ctx.set_particles(x, v, m)
    return p, ctx


def update(ctx, F, rng):
    n = ctx.n
    ins = {"F": F, "c": rng.uniform(0.3, 1.0, n), "g": rng.uniform(0.1, 1.0, n),
           "alpha": rng.uniform(0.0, 0.9, n), "psi": np.zeros(n)}
    ins = {k: a.astype(np.float32).astype(np.float64) for k, a in ins.items()}
    for k, a in ins.items():
        ctx.set(k, a)
    ctx.stress()
    return ins


def bounds(F):
    s = np.linalg.svd(F, compute_uv=False)
    return 1e-6 + 1.8e-7 * np.abs(np.log(s)).max(axis=1) + 3e-14 * s[:, 0] / s[:, 2]


def compare(ctx, ref, keys, bound, use):
    for k in keys:
        got = ctx.get(k).reshape(ctx.n, -1)[use]
        want = np.array([np.ravel(r[k]) for r in ref])[use]
        scale = np.abs(want).max(axis=1) + 1e-30
        err = np.abs(got - want).max(axis=1) / scale / bound[use]
        assert err.max() < 1.0, (k, err.max())


@pytest.mark.parametrize("kind", KINDS)
def test_volume(mpmx, oracle, kind):
    p, ctx = setup(mpmx, 2)
    ins = update(ctx, gradients(kind, ctx.n, np.random.default_rng(21)), np.random.default_rng(22))
    op = oracle_params(oracle, p)
    ref = [oracle.von_mises(op, ins["F"][i], ins["c"][i], ins["g"][i], ins["alpha"][i], 0.0) for i in range(ctx.n)]
    use = np.array([np.isfinite(r["sigma"]).all() for r in ref])
    assert use.mean() > 0.2
    compare(ctx, ref, ["vol"], bounds(ins["F"]), use)


@pytest.mark.parametrize("kind", KINDS)
def test_neo_hookean(mpmx, oracle, kind):
    p, ctx = setup(mpmx, 1)
    ins = update(ctx, gradients(kind, ctx.n, np.random.default_rng(23)), np.random.default_rng(24))
    op = oracle_params(oracle, p)
    ref = [oracle.neo_hookean(op, ins["F"][i], ins["c"][i], 0.0) for i in range(ctx.n)]
    use = np.array([np.isfinite(r["sigma"]).all() for r in ref])
    if "reflected" in kind:   # no energy at J < 0
        assert not use.any()
        with pytest.raises(mpmx.MpmxError) as e:
            ctx.sync()
        assert e.value.status == mpmx.ERR_NONFINITE
        return
    assert use.all()
    # psi itself, the difference of a shear and a volume part, shows the rounding of
    # their constants wherever the two cancel; FP holds it in the way it is used
    compare(ctx, ref, ["sigma", "FP", "vol"], bounds(ins["F"]), use)
    assert np.array_equal(ctx.get("F"), ins["F"])


@pytest.mark.parametrize("kind", KINDS + ["flat"])
def test_fixed_corotated(mpmx, oracle, kind):
    p, ctx = setup(mpmx, 0)
    ins = update(ctx, gradients(kind, ctx.n, np.random.default_rng(25)), np.random.default_rng(26))
    op = oracle_params(oracle, p)
    ref = [{"sigma": oracle.fixed_corotated(op, F), "vol": p.V0 * np.linalg.det(F)} for F in ins["F"]]
    use = np.ones(ctx.n, bool)
    compare(ctx, ref, ["sigma"], np.full(ctx.n, 1e-6), use)
    if kind != "flat":
        compare(ctx, ref, ["vol"], bounds(ins["F"]), use)
    assert np.array_equal(ctx.get("F"), ins["F"])


def lower_rank(rank, n, rng):
    """Sums of `rank` products of small integers, exact in FP32; the largest singular
    value is above 2, far past the yield strain whatever the others are taken for."""
    a = rng.integers(1, 9, (n, 3, rank)) * rng.choice([-1, 1], (n, 3, rank))
    b = rng.integers(1, 9, (n, 3, rank)) * rng.choice([-1, 1], (n, 3, rank))
    return (a @ b.transpose(0, 2, 1)) / 4.0 if rank else np.zeros((n, 3, 3))


@pytest.mark.parametrize("rank", [0, 1, 2])
def test_lower_rank(mpmx, oracle, rank):
    """Fixed corotated stress has a value at any rank.  Under von Mises the smallest
    singular values are rounding noise and so is the flow, but F and the stress are
    finite; F = 0 does not flow and has no energy."""
    p, ctx = setup(mpmx, 0)
    ins = update(ctx, lower_rank(rank, ctx.n, np.random.default_rng(27)), np.random.default_rng(28))
    op = oracle_params(oracle, p)
    ref = [{"sigma": oracle.fixed_corotated(op, F)} for F in ins["F"]]
    compare(ctx, ref, ["sigma"], np.full(ctx.n, 1e-6), np.ones(ctx.n, bool))
    p, ctx = setup(mpmx, 2)
    ins = update(ctx, lower_rank(rank, ctx.n, np.random.default_rng(27)), np.random.default_rng(28))
    if rank == 0:
        with pytest.raises(mpmx.MpmxError) as e:
            ctx.sync()
        assert e.value.status == mpmx.ERR_NONFINITE
        return
    F = ctx.get("F")
    assert np.isfinite(F).all() and np.isfinite(ctx.get("sigma")).all()
    assert (F != ins["F"]).any(axis=(1, 2)).all()
