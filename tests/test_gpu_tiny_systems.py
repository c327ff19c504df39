"""Exact ensembles whose largest system has few bodies: none, one or an odd number of sources, in few and many wavefronts."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [2], [2, 1], [3], [3, 1, 2], [4], [5], [7, 2], [9]])
@pytest.mark.parametrize("flags", [A.NEWTON, A.NEWTON | A.PN1, A.NEWTON | A.EIH])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 120])
def test_bits_of_the_oracle(ctx, orc, sizes, flags, scale):
    """Leapfrog and (Newtonian) Wisdom-Holman, inside the ranges of the short exact forms and beyond them."""
    rng = np.random.default_rng(len(sizes) + sizes[0])
    n = sum(sizes)
    pos, vel = scale * rng.normal(size=(n, 3)), 0.1 * rng.normal(size=(n, 3))
    mass = rng.uniform(0.5, 1.5, n)
    first = np.concatenate([[0], np.cumsum(sizes)])
    runs = [(A.LEAPFROG, 1e-2 * scale)]
    if flags == A.NEWTON and scale == 1.0:
        runs.append((A.WH_PLANETARY, 1e-3))
    for integrator, dt in runs:
        m = mass.copy()
        if integrator == A.WH_PLANETARY:
            m *= 1e-3
            m[first[:-1]] = 1.0
        for copies in (1, -(-64 * 1100 // n)):
            ctx.set_params(G=1.1, softening=0.0, c=20.0, pn_flags=flags, precision=A.FP64)
            off = np.concatenate([[0], np.cumsum(sizes * copies)]).astype(np.int64)
            ctx.batch_set(off, np.tile(pos, (copies, 1)), np.tile(vel, (copies, 1)), np.tile(m, copies))
            ctx.batch_step(integrator, dt, 3)
            p, v = (x.reshape(copies, n, 3) for x in ctx.batch_get())
            assert np.array_equal(p, np.broadcast_to(p[0], p.shape)) and np.array_equal(v, np.broadcast_to(v[0], v.shape))
            for a, b in zip(first[:-1], first[1:]):
                if integrator == A.WH_PLANETARY:
                    rp, rv = orc.integrate_wh(pos[a:b], vel[a:b], m[a:b], dt, 3, G=1.1)
                else:
                    rp, rv, _ = orc.integrate(pos[a:b], vel[a:b], m[a:b], dt, 3, integrator=2, G=1.1, c=20.0, soft=0.0,
                                              pn=flags)
                assert np.array_equal(p[0, a:b], rp) and np.array_equal(v[0, a:b], rv), (integrator, copies, a)


@pytest.mark.parametrize("largest", [3, 6, 10, 13, 24, 58])
@pytest.mark.parametrize("flags", [A.NEWTON, A.NEWTON | A.PN1])
@pytest.mark.parametrize("precision", [A.FP64, A.FP32])
def test_same_bits_whatever_shares_the_chip(ctx, largest, flags, precision):
    """Systems of one size and of falling sizes in up to five rounds of 256 wavefronts: the bits of the same systems in more
    wavefronts than teams take."""
    rng = np.random.default_rng(largest)
    pos, vel = rng.normal(size=(largest, 3)), 0.3 * rng.normal(size=(largest, 3))
    mass = 10.0 ** rng.uniform(-3.0, 0.0, largest)
    per = 64 // largest
    ctx.set_params(G=1.2, softening=1e-3, c=20.0, pn_flags=flags, precision=precision)

    def run(sizes):
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
        take = np.concatenate([np.arange(k) for k in sizes])
        ctx.batch_set(off, pos[take], vel[take], mass[take])
        ctx.batch_step(A.LEAPFROG, 1e-2, 3)
        p, v = ctx.batch_get()
        return {int(k): (p[a:a + k], v[a:a + k]) for a, k in zip(off[:-1][::-1], sizes[::-1])}

    ref = run([largest, 3, 2] * (per * 1300))
    for waves in (200, 400, 600, 900):
        small = [3, 2] * (8 * waves)
        for sizes in ([largest] * (per * waves), [largest] * (per * 256) + small, [largest] * (per * 256 + 1) + [3] * 700):
            for k, (p, v) in run(sizes).items():
                assert np.array_equal(p, ref[k][0]) and np.array_equal(v, ref[k][1]), (waves, len(sizes), k)
