"""What a trajectory gradient's two passes leave and expect: systems loaded, parameters changed or steps taken between or
after them."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


def systems(sizes, seed=1):
    n, rng = sum(sizes), np.random.default_rng(seed)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    return off, rng.normal(size=(n, 3)), 0.1 * rng.normal(size=(n, 3)), rng.uniform(0.5, 1.5, n)


@pytest.mark.parametrize("sizes", [[3] * 4, [3] * 400, [5, 2, 64], [3]])
def test_loading_systems_drops_the_stored_trajectory(ctx, sizes):
    """The backward pass refuses (on the host) after other systems, fewer or more, were loaded."""
    ctx.set_params(G=1.0, softening=1e-2)
    ctx.batch_set(*systems([3] * 4))
    ctx.batch_traj_forward(1e-2, 4, [4])
    e = systems(sizes, 2)
    ctx.batch_set(*e)
    with pytest.raises(A.AsterError) as err:
        ctx.batch_traj_backward(np.zeros((1, sum(sizes), 3)))
    assert err.value.code == -6  # ASTER_ERR_STATE
    p, v = ctx.batch_get()
    assert np.array_equal(p, e[1]) and np.array_equal(v, e[2])


@pytest.mark.parametrize("precision", [A.FP64, A.FP32])
@pytest.mark.parametrize("sizes", [[3] * 40, [1, 2, 3, 17, 64]])
def test_steps_after_a_forward_pass(ctx, orc, sizes, precision):
    """They begin with an evaluation of their own: the bits of the same state loaded afresh, in the exact mode those of the
    oracle."""
    off, pos, vel, mass = systems(sizes)
    ctx.set_params(G=1.1, softening=1e-2, precision=precision)
    ctx.batch_set(off, pos, vel, mass)
    ctx.batch_step(A.LEAPFROG, 1e-2, 2)
    ctx.batch_traj_forward(1e-2, 3, [3])
    p0, v0 = ctx.batch_get()
    ctx.batch_step(A.LEAPFROG, 1e-2, 4)
    p, v = ctx.batch_get()
    ctx.batch_set(off, p0, v0, mass)
    ctx.batch_step(A.LEAPFROG, 1e-2, 4)
    q, w = ctx.batch_get()
    assert np.array_equal(p, q) and np.array_equal(v, w)
    if precision == A.FP64:
        for a, b in zip(off[:-1], off[1:]):
            rp, rv, _ = orc.integrate(p0[a:b], v0[a:b], mass[a:b], 1e-2, 4, integrator=2, G=1.1, soft=1e-2)
            assert np.array_equal(p[a:b], rp) and np.array_equal(v[a:b], rv)


@pytest.mark.parametrize("changed", [dict(G=2.5), dict(softening=0.3), dict(theta=0.9)])
@pytest.mark.parametrize("ensemble", [False, True])
def test_parameters_set_between_the_passes(ctx, changed, ensemble):
    """The gradient is that of the trajectory as it was run, and what follows uses the new parameters."""
    off, pos, vel, mass = systems([3] * 30 + [17])
    n = len(mass)
    rng = np.random.default_rng(5)
    g = rng.normal(size=(2, n, 3))
    out = []
    for change in (False, True):
        ctx.set_params(G=1.0, softening=1e-2, theta=0.5)
        if ensemble:
            ctx.batch_set(off, pos, vel, mass)
            ctx.batch_traj_forward(1e-2, 6, [3, 6])
        else:
            ctx.set_state(pos, vel, mass)
            ctx.traj_forward(1e-2, 6, 4, [3, 6])
        if change:
            ctx.set_params(**changed)
        out.append(ctx.batch_traj_backward(g) if ensemble else ctx.traj_backward(g))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert all(getattr(ctx.params(), k) == v for k, v in changed.items())
    if ensemble or "theta" in changed:  # (without a new force law the backward pass's accelerations serve the next step)
        return
    ctx.step(A.ALLPAIRS_FP32_KAHAN, A.LEAPFROG, 1e-2, 1)
    p, _ = ctx.get_state()
    ctx.set_state(pos, vel, mass)
    ctx.step(A.ALLPAIRS_FP32_KAHAN, A.LEAPFROG, 1e-2, 1)
    assert np.array_equal(p, ctx.get_state()[0])


@pytest.mark.parametrize("n", [100, 5000])
def test_evaluations_between_the_passes(ctx, n):
    """Accelerations of another method, force law or source range do not enter the time reversal, nor are those of the
    backward pass taken for the range's."""
    pos, vel, mass = A.ic_plummer(n, 2)
    g = np.random.default_rng(5).normal(size=(1, n, 3))
    out = []
    for between in (None, dict(lower=n // 2), dict(G=3.0)):
        ctx.set_params(G=1.0, softening=1e-2, theta=0.8, lower=0)
        ctx.set_state(pos, vel, mass)
        ctx.traj_forward(1e-2, 6, 4, [6])
        if between:
            ctx.forces(A.BH_GROUP, out=False)
            ctx.set_params(**between)
            ctx.forces(A.ALLPAIRS_FP32_KAHAN, out=False)
        out.append(ctx.traj_backward(g))
        for a, b in zip(out[0], out[-1]):
            assert np.array_equal(a, b), between
        if between:
            ctx.step(A.ALLPAIRS_FP32_KAHAN, A.LEAPFROG, 1e-2, 1)
            p, _ = ctx.get_state()
            ctx.set_state(pos, vel, mass)
            ctx.step(A.ALLPAIRS_FP32_KAHAN, A.LEAPFROG, 1e-2, 1)
            assert np.array_equal(p, ctx.get_state()[0])
