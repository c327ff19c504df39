"""Source ranges of the all-pairs methods at the ends of the body arrays, on each side of the lines between kernels."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 4096, 4097, 26624, 32768, 65536, 65537])
@pytest.mark.parametrize("method", [A.ALLPAIRS_FP32_KAHAN, A.ALLPAIRS_FP32, A.ALLPAIRS_FP64])
def test_empty_source_range(ctx, n, method):
    """No source: zero accelerations, also behind the last body of an array without padding, and after a larger state
    whose records lie behind this one's."""
    for bodies in (n + 300, n):
        pos, vel, mass = A.ic_cube(bodies, 3)
        ctx.set_params(G=1.0, softening=1e-3, lower=0, upper=-1)
        ctx.set_state(pos, vel, mass)
        ctx.forces(method, out=False)
    for at in (0, n // 2, n - 1, n):
        for soft in (1e-3, 0.0):
            ctx.set_params(softening=soft, lower=at, upper=at)
            assert not np.any(ctx.forces(method)), (at, soft)


@pytest.mark.parametrize("n", [4096, 26625, 32769])
@pytest.mark.parametrize("method", [A.ALLPAIRS_FP32_KAHAN, A.ALLPAIRS_FP32])
def test_last_bodies_as_sources(ctx, n, method):
    """The last body and the last bodies across a tile's edge, against FP64 (bars of the FP32 methods)."""
    pos, vel, mass = A.ic_cube(n, 4)
    bar = 1e-5 if method == A.ALLPAIRS_FP32_KAHAN else 1e-4
    for lower in (n - 1, n - 65):
        ctx.set_params(G=1.0, softening=1e-2, lower=lower, upper=n)
        ctx.set_state(pos, vel, mass)
        ref = ctx.forces(A.ALLPAIRS_FP64)
        err = np.linalg.norm(ctx.forces(method) - ref, axis=1)
        scale = np.linalg.norm(ref, axis=1)
        assert np.all(err <= bar * np.maximum(scale, np.median(scale)))
