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
