"""The all-pairs FP32 paths over small and middle sizes, through the C ABI: the
sizes at which the kernel, the number of rounds or the last tile changes. The
updates fused into the evaluation give the bits of separate calls."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu

SIZES = [1, 15, 16, 17, 64, 65, 1000, 1024, 1025, 2112, 4095, 4096, 4097, 20481, 32768, 32769]


def state(n, seed=3):
    pos, vel, mass = A.ic_plummer(n, seed, mass_mode=1)
    return pos, vel, mass


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("soft", [2.5e-5, 0.0])
def test_fp32_forces_against_fp64(ctx, n, soft):
    """The FP32 bars (mixed 1e-5, plain 1e-4) of every body relative to max(|a_i|, median |a|), full range and a source
    range that starts and ends inside tiles."""
    pos, vel, mass = state(n)
    ranges = [(0, -1)] + ([(n // 3, n - n // 5)] if n > 10 else [])
    for lower, upper in ranges:
        ctx.set_params(G=1.3, softening=soft, lower=lower, upper=upper)
        ctx.set_state(pos, vel, mass)
        ref = ctx.forces(A.ALLPAIRS_FP64)
        scale = np.linalg.norm(ref, axis=1)
        scale = np.maximum(scale, np.median(scale)) + 1e-300
        for method, bar in ((A.ALLPAIRS_FP32_KAHAN, 1e-5), (A.ALLPAIRS_FP32, 1e-4)):
            err = np.linalg.norm(ctx.forces(method) - ref, axis=1) / scale
            assert err.max() <= bar, (lower, upper, method, err.max())


@pytest.mark.parametrize("n", [1, 17, 1025, 4096, 4097, 33000])
@pytest.mark.parametrize("method", [A.ALLPAIRS_FP32_KAHAN, A.ALLPAIRS_FP32])
def test_fused_updates_same_bits_as_separate_calls(ctx, n, method):
    """Several steps in one call against one step per call (whose closing kick and opening drift are launches of their
    own), for every integrator, with and without velocity-dependent terms."""
    pos, vel, mass = state(n)
    runs = [(A.LEAPFROG, 0, A.NEWTON), (A.YOSHIDA4, 0, A.NEWTON), (A.EULER, 1, A.NEWTON), (A.SABA, 3, A.NEWTON)]
    if n < 5000:
        runs.append((A.LEAPFROG, 0, A.NEWTON | A.PN1))
    for integrator, order, flags in runs:
        out = []
        for parts in ((3,), (1, 1, 1)):
            ctx.set_params(G=1.0, softening=1e-4, c=10.0, pn_flags=flags)
            ctx.set_state(pos, vel, mass)
            for k in parts:
                ctx.integrate(method, integrator, order, 1e-3, k)
            out.append(ctx.get_state() + (ctx.get_acc(),))
        for a, b in zip(*out):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b), (integrator, order, flags)


@pytest.mark.parametrize("n", [2, 16, 17, 100, 1025, 4097])
def test_gradient_against_oracle(ctx, orc, n):
    """Relative 2-norm of each gradient block against the FP64 oracle adjoint: 1e-4, the bar of the adjoint's own tests."""
    pos, vel, mass = A.ic_plummer(n, 5)
    steps, snaps = (12, [4, 5, 12]) if n < 1000 else (4, [1, 4])
    rng = np.random.default_rng(n)
    ctx.set_params(G=1.0, softening=1e-2)
    ctx.set_state(pos, vel, mass)
    s = ctx.traj_forward(1e-2, steps, 4 if n < 1000 else 3, snaps)
    target = s + rng.normal(scale=1e-2, size=s.shape)
    got = ctx.traj_backward(2.0 * (s - target) / (n * len(snaps)))
    _, *ref = orc.traj_grad(pos, vel, mass, 1e-2, steps, np.array(snaps), target, soft=1e-2)
    for g, r in zip(got, ref):
        assert np.linalg.norm(g - r) <= 1e-4 * np.linalg.norm(r)
    p, v = ctx.get_state()
    assert np.array_equal(p, pos) and np.array_equal(v, vel)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 8192, 8193, 8300])
@pytest.mark.parametrize("soft", [1e-4, 0.0])
def test_energy_against_oracle(ctx, orc, n, soft):
    """One tile, its edges, one tile per strip and the first longer strips: 1e-12 relative, the bar of the energy's own
    test (sums in another order), and the same bits on a second call."""
    pos, vel, mass = state(n)
    ctx.set_params(G=1.3, softening=soft)
    ctx.set_state(pos, vel, mass)
    e, ep, L = ctx.energy()
    re, rep, rL = orc.energy(pos, vel, mass, G=1.3, soft=soft)
    kin = 0.5 * float((mass[:, None] * vel * vel).sum())  # e is kinetic minus potential: bound by the larger part
    assert abs(e - re) <= 1e-12 * (abs(re) + 2 * kin) and abs(ep - rep) <= 1e-12 * (abs(rep) + 2 * kin)
    np.testing.assert_allclose(L, rL, rtol=1e-10, atol=1e-14)
    e2, ep2, L2 = ctx.energy()
    assert (e, ep) == (e2, ep2) and np.array_equal(L, L2)


@pytest.mark.parametrize("n", [4, 37, 64, 65, 66, 200, 1500])
@pytest.mark.parametrize("soft", [2.5e-5, 0.0])
@pytest.mark.parametrize("flags", [A.NEWTON | A.PN1, A.NEWTON | A.PN1 | A.PN25])
def test_group_traversal_pn_small_groups(ctx, orc, n, soft, flags):
    """Post-Newtonian part of the group traversal at the edges of groups, pieces and list batches, with two bodies at one
    place: against the oracle's lists, the bars of the traversal's own test."""
    pos, vel, mass = A.ic_mixed(n, n)
    pos[n // 2] = pos[0]
    part = []
    for f in (A.NEWTON, flags):
        ctx.set_params(G=1.0, softening=soft, theta=0.6, c=30.0, pn_flags=f)
        ctx.set_state(pos, vel, mass)
        part.append(ctx.forces(A.BH_GROUP))
    ref = orc.bh_group_pn(pos, vel, mass, orc.box_auto(pos), 0.6, c=30.0, soft=soft, pn=flags)
    scale = np.linalg.norm(ref, axis=1)
    err = np.linalg.norm(part[1] - part[0] - ref, axis=1)
    assert np.all(err <= 1e-9 * np.maximum(scale, np.median(scale)) + 1e-15 * np.abs(part[1]).max())


@pytest.mark.parametrize("sizes", [[1], [2], [3], [3] * 16, [3] * 50, [4] * 20, [1, 2, 3, 4, 5, 8, 21, 32, 33, 63, 64]])
@pytest.mark.parametrize("snaps", [[1, 2, 7], [4], [9, 10]])
def test_batch_gradient_against_oracle(ctx, orc, sizes, snaps):
    """Odd and even systems, alone and packed, more and fewer steps than are loaded ahead: the bars of the three-body test."""
    n, steps = sum(sizes), snaps[-1] + (len(snaps) == 3)
    rng = np.random.default_rng(n)
    pos, vel = rng.normal(size=(n, 3)), 0.1 * rng.normal(size=(n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    off = np.concatenate([[0], np.cumsum(sizes)])
    ctx.set_params(G=1.3, softening=1e-2, precision=A.FP32)
    ctx.batch_set(off, pos, vel, mass)
    s = ctx.batch_traj_forward(1e-2, steps, snaps)
    target = s + rng.normal(scale=1e-2, size=s.shape)
    gsnap = 2.0 * (s - target)
    got = ctx.batch_traj_backward(gsnap)
    p, v = ctx.batch_get()
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    for a, b in zip(off[:-1], off[1:]):
        loss, *ref = orc.traj_grad(pos[a:b], vel[a:b], mass[a:b], 1e-2, steps, np.array(snaps), target[:, a:b], G=1.3, soft=1e-2)
        assert loss * (b - a) * len(snaps) == pytest.approx(((s - target)[:, a:b] ** 2).sum(), rel=1e-10)
        for g, r in zip(got, ref):
            assert np.linalg.norm(g[a:b] - r * (b - a) * len(snaps)) <= 1e-8 * np.linalg.norm(r) * (b - a) * len(snaps)


@pytest.mark.parametrize("largest", [2, 4, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("flags", [A.NEWTON, A.NEWTON | A.PN1])
@pytest.mark.parametrize("precision", [A.FP64, A.FP32])
def test_ensembles_same_bits_whatever_their_number(ctx, largest, flags, precision):
    """A few systems, a few hundred wavefronts and more wavefronts than the teams take: the same systems give the same
    bits (each rule's kernel against the one for large ensembles, itself tested against the oracle)."""
    rng = np.random.default_rng(largest)
    sizes = [largest] + [int(k) for k in rng.integers(1, largest + 1, 6)]
    n = sum(sizes)
    pos, vel = rng.normal(size=(n, 3)), 0.3 * rng.normal(size=(n, 3))
    mass = 10.0 ** rng.uniform(-3.0, 0.0, n)
    out = []
    for waves in (1, 300, 450, 1100):
        k = -(-64 * waves // n)
        off = np.concatenate([[0], np.cumsum(sizes * k)])
        ctx.set_params(G=1.2, softening=1e-3, c=20.0, pn_flags=flags, precision=precision)
        ctx.batch_set(off, np.tile(pos, (k, 1)), np.tile(vel, (k, 1)), np.tile(mass, k))
        ctx.batch_step(A.YOSHIDA4, 1e-2, 2)
        ctx.batch_step(A.LEAPFROG, 1e-2, 3)
        p, v = ctx.batch_get()
        assert np.array_equal(p, np.tile(p[:n], (k, 1))) and np.array_equal(v, np.tile(v[:n], (k, 1))), waves
        out.append((p[:n], v[:n]))
    for p, v in out:
        assert np.all(np.isfinite(p)) and np.array_equal(p, out[-1][0]) and np.array_equal(v, out[-1][1])


@pytest.mark.parametrize("n", [26624, 26625])
def test_fp32_forces_at_the_mixed_line(ctx, n):
    """Both sides of the line between the mixed method's kernels: the bars of the other sizes, and fused updates."""
    test_fp32_forces_against_fp64(ctx, n, 2.5e-5)
    test_fused_updates_same_bits_as_separate_calls(ctx, n, A.ALLPAIRS_FP32_KAHAN)
