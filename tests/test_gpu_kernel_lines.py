"""Lines between kernels that other tests do not stand at."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


def test_gradient_at_the_line_of_its_kernels(ctx):
    """20480 bodies are the last that the adjoint takes from LDS: with one more of next to no mass, far away, the other
    kernel gives the same gradients to 1e-4 in the 2-norm of each block, the bar of the adjoint's own tests."""
    n, steps, snaps = 20480, 3, [1, 3]
    pos, vel, mass = A.ic_plummer(n, 5)
    g = np.random.default_rng(1).normal(size=(2, n, 3))
    out = []
    for extra in (0, 1):
        p, v = np.vstack([pos, np.full((extra, 3), 1e3)]), np.vstack([vel, np.zeros((extra, 3))])
        ctx.set_params(G=1.0, softening=1e-2)
        ctx.set_state(p, v, np.concatenate([mass, np.full(extra, 1e-12)]))
        s = ctx.traj_forward(1e-2, steps, 2, snaps)
        grads = ctx.traj_backward(np.concatenate([g, np.zeros((2, extra, 3))], 1))
        q, w = ctx.get_state()
        assert np.array_equal(q, p) and np.array_equal(w, v)
        out.append([s[:, :n]] + [x[:n] for x in grads])
    for a, b in zip(*out):
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(a)


@pytest.mark.parametrize("n", [1, 17, 1000, 8193, 16384, 16385])
@pytest.mark.parametrize("integrator,order", [(A.LEAPFROG, 0), (A.SABA, 3)])
def test_fp64_source_range_past_the_last_body(ctx, n, integrator, order):
    """A source range that ends behind the last body is all of them: the same bits, with the update fused or not."""
    pos, vel, mass = A.ic_plummer(n, 4, mass_mode=1)
    out = []
    for upper in (-1, n + 1):
        ctx.set_params(G=1.0, softening=1e-4, lower=0, upper=upper)
        ctx.set_state(pos, vel, mass)
        ctx.integrate(A.ALLPAIRS_FP64, integrator, order, 1e-3, 2)
        out.append(ctx.get_state() + (ctx.get_acc(),))
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
