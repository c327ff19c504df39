"""The moments of trees of more than 2^21 bodies, whose largest nodes are formed in a launch more."""
import numpy as np
import pytest

import aster_amd as A

pytestmark = pytest.mark.gpu


def bodies(n, chains):
    """Uniform above z = 0; below, 25 clusters of 8300 bodies in one Morton cell each, with 24 bodies that split off one by
    one: more than 512 nodes of more than 8192 leaves in a half of the tree."""
    rng = np.random.default_rng(n)
    cells = []
    for p in (rng.permutation(32)[:25] if chains else []):
        cell = np.array([p & 3, p >> 2 & 3, p >> 4]) * 256 + rng.integers(0, 256, 3)
        cells += [cell] * 8300
        for j in range(8):
            for axis in range(3):
                c = cell.copy()
                c[axis] ^= 1 << j
                cells.append(c)
    low = (np.array(cells).reshape(-1, 3) + rng.uniform(0.1, 0.9, (len(cells), 3))) / 512.0 - 1.0
    pos = np.concatenate([low, rng.uniform([-1.0, -1.0, 0.0 if chains else -1.0], 1.0, (n - len(low), 3))])
    pos = pos[rng.permutation(n)]
    return pos, 0.1 * rng.normal(size=(n, 3)), rng.uniform(0.5, 1.5, n) / n


@pytest.mark.parametrize("n,chains", [((1 << 21) + 1, False), (2400000, True), (5000011, False)])
def test_every_node_from_its_children(ctx, n, chains):
    """A node's mass and centre are the bits of the two children's (and so, upwards from the leaves, of the whole tree's);
    forces of some bodies against direct sums: 1e-2 of the median, as an opening angle of 0.4 gives, to see that the boxes
    of the large nodes are there."""
    pos, vel, mass = bodies(n, chains)
    ctx.set_params(G=1.0, softening=1e-3, theta=0.4, box=(1.0, 1.0, 1.0))
    ctx.set_state(pos, vel, mass)
    acc = ctx.forces(A.BH_GROUP)
    t = ctx.tree()
    assert np.array_equal(t["mass"][:n], mass[t["perm"]]) and np.array_equal(t["com"][:n], pos[t["perm"]])
    L, R = t["left"][n:], t["right"][n:]
    mL, mR = t["mass"][L], t["mass"][R]
    assert np.array_equal(t["mass"][n:], mR + mL)
    for c in range(3):
        x = t["com"][:, c]
        assert np.array_equal(x[n:], (x[R] * mR + x[L] * mL) / (mR + mL))
    some, ref = np.random.default_rng(1).integers(0, n, 24), []
    for i in some:
        d = pos - pos[i]
        w = mass * ((d * d).sum(1) + 1e-3) ** -1.5
        ref.append((w[:, None] * d).sum(0))
    err, scale = np.linalg.norm(acc[some] - ref, axis=1), np.linalg.norm(ref, axis=1)
    assert np.all(err <= 1e-2 * np.maximum(scale, np.median(scale))), (err / scale).max()


@pytest.mark.parametrize("n,chains", [((1 << 21) + 1, False), (2400000, True)])
def test_velocities_of_the_nodes(ctx, orc, n, chains):
    """The FP64 traversal with 1PN terms reads every node's velocity: the oracle's bits."""
    pos, vel, mass = bodies(n, chains)
    ctx.set_params(G=1.0, softening=1e-3, theta=0.8, c=2.0, box=(1.0, 1.0, 1.0), pn_flags=A.NEWTON | A.PN1,
                   precision=A.FP64)
    ctx.set_state(pos, vel, mass)
    ref = orc.bh(pos, vel, mass, np.ones(3), 0.8, c=2.0, soft=1e-3, pn=A.NEWTON | A.PN1)
    assert np.array_equal(ctx.forces(A.BH_PARITY), ref)
