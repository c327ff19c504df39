"""The Morton sort where the tiles' digit counts are summed by groups and those scanned: both sides of the lines."""
import ctypes

import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, (1 << 21) + 1, (1 << 21) + 131073, 5000011])
def test_sorted_codes_and_order(ctx, n):
    """Codes ascending, equal ones in body order, every body once; a third of the bodies shares some hundred cells."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(-1.0, 1.0, (n, 3))
    k = n // 3
    pos[rng.permutation(n)[:k]] = rng.uniform(-1.0, 1.0, (900, 3))[rng.integers(0, 900, k)]
    ctx.set_params(G=1.0, softening=1e-2, theta=1.0, box=(1.0, 1.0, 1.0))
    ctx.set_state(pos, None, np.full(n, 1.0 / n))
    codes, _ = ctx.morton()
    ctx.forces(A.BH_GROUP, out=False)
    got, perm = np.empty(n, np.uint32), np.empty(n, np.uint32)
    u32 = ctypes.POINTER(ctypes.c_uint32)
    assert A.lib().aster_tree_dump(ctx.h, got.ctypes.data_as(u32), perm.ctypes.data_as(u32), None, None, None, None) == 0
    assert np.array_equal(np.bincount(perm, minlength=n), np.ones(n))
    assert np.array_equal(codes[perm], got)
    up, same = got[1:] > got[:-1], got[1:] == got[:-1]
    assert np.all(up | (same & (perm[1:] > perm[:-1]))) and np.count_nonzero(same) > k // 2
