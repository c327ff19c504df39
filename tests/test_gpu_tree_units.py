"""Moments above the traversal groups where a workgroup has more nodes than threads, and the walk's stack at its limit."""
import numpy as np
import pytest

import aster_amd as A

BOX = np.ones(3)


def chains(nclusters, core, seed=1):
    """Clusters of `core` bodies in one Morton cell, each with 24 bodies that split off it one by one: every one of the
    24 levels above the core has a node with a single-body group on one side."""
    rng = np.random.default_rng(seed)
    cells, places = [], rng.permutation(64)[:nclusters]
    for p in places:
        cell = np.array([p & 3, p >> 2 & 3, p >> 4]) * 256 + rng.integers(0, 256, 3)
        cells += [cell] * core
        for j in range(8):
            for axis in range(3):
                c = cell.copy()
                c[axis] ^= 1 << j
                cells.append(c)
    pos = (np.array(cells) + rng.uniform(0.1, 0.9, (len(cells), 3))) / 512.0 - 1.0
    vel = rng.normal(size=pos.shape)
    mass = rng.uniform(0.5, 1.5, len(pos)) / len(pos)
    order = rng.permutation(len(pos))
    return pos[order], vel[order], mass[order]


def sizes(left, right, n):
    """Leaves below every node."""
    size = np.zeros(2 * n - 1, np.int64)
    stack = [(n, False)]
    while stack:
        node, ready = stack.pop()
        if node < n:
            size[node] = 1
        elif ready:
            size[node] = size[left[node]] + size[right[node]]
        else:
            stack += [(node, True), (int(left[node]), False), (int(right[node]), False)]
    return size


# one unit of ~1000 groups; several such units; more than 512 nodes above the units
CASES = [(40, 66, 256, 0), (60, 130, 256, 0), (25, 4150, 0, 512)]


@pytest.mark.parametrize("nclusters,core,in_unit,top", CASES)
def test_inputs_exceed_the_threads(orc, nclusters, core, in_unit, top):
    pos, vel, mass = chains(nclusters, core)
    n = len(mass)
    t = orc.build_tree(pos, vel, mass, BOX)
    left, right = t["left"], t["right"]
    size = sizes(left, right, n)
    assert np.count_nonzero(size > 4096) >= top
    most = 0
    roots = [n] if n <= 4096 else [k for p in np.flatnonzero(size > 4096) for k in (left[p], right[p])]
    for r in roots:
        if 64 < size[r] <= 4096:
            count, stack = 0, [int(r)]
            while stack:
                k = stack.pop()
                if size[k] > 64:
                    count += 1
                    stack += [int(left[k]), int(right[k])]
            most = max(most, count)
    assert most > in_unit or in_unit == 0


# more than 512 nodes above units of 8192 leaves; units of that size with more than 512 nodes
CASES8 = [(25, 8300, 0, 512), (60, 130, 512, 0)]


@pytest.mark.parametrize("nclusters,core,in_unit,top", CASES8)
def test_inputs_exceed_the_threads_of_larger_units(orc, nclusters, core, in_unit, top):
    pos, vel, mass = chains(nclusters, core)
    n = len(mass)
    t = orc.build_tree(pos, vel, mass, BOX)
    size = sizes(t["left"], t["right"], n)
    big = np.flatnonzero(size > 8192)
    assert len(big) >= top
    inside = [sum(1 for k in subtree(t, r) if size[k] > 64) for p in big for r in (t["left"][p], t["right"][p])
              if 64 < size[r] <= 8192]
    assert max(inside) > in_unit


def subtree(t, root):
    stack = [int(root)]
    while stack:
        k = stack.pop()
        yield k
        if t["left"][k] >= 0:
            stack += [int(t["left"][k]), int(t["right"][k])]


@pytest.mark.gpu
@pytest.mark.parametrize("nclusters,core,in_unit,top", CASES + CASES8[:1])
def test_moments_of_many_nodes(ctx, orc, nclusters, core, in_unit, top):
    """The tree's bits for each traversal, the lists, and the velocity moments through the post-Newtonian part (bars of the
    traversal's own tests)."""
    pos, vel, mass = chains(nclusters, core)
    ref = orc.build_tree(pos, vel, mass, BOX)
    ctx.set_params(G=1.0, softening=1e-3, theta=0.5, c=30.0, box=(1.0, 1.0, 1.0))
    ctx.set_state(pos, vel, mass)
    for method in (A.BH_GROUP, A.BH_PARITY):
        ctx.forces(method, out=False)
        tree = ctx.tree()
        for key in ("codes", "perm", "left", "right", "mass", "com"):
            assert np.array_equal(tree[key], ref[key]), (method, key)
    ctx.bh_stats()
    newton = ctx.forces(A.BH_GROUP)
    _, inter, visits = orc.bh_group(pos, mass, BOX, 0.5, soft=1e-3)
    assert ctx.bh_stats() == (inter, visits)
    ctx.set_params(G=1.0, softening=1e-3, theta=0.5, c=30.0, box=(1.0, 1.0, 1.0), pn_flags=A.NEWTON | A.PN1)
    both = ctx.forces(A.BH_GROUP)
    pn = orc.bh_group_pn(pos, vel, mass, BOX, 0.5, c=30.0, soft=1e-3, pn=A.NEWTON | A.PN1)
    scale = np.linalg.norm(pn, axis=1)
    err = np.linalg.norm(both - newton - pn, axis=1)
    assert np.all(err <= 1e-9 * np.maximum(scale, np.median(scale)) + 1e-15 * np.abs(both).max())


@pytest.mark.gpu
def test_stack_at_its_limit(ctx):
    """Opening angle 0 opens every node: 32 entries wait per level, so from ~2^15 bodies on the walk reaches the stack's
    limit and narrows. Every pair is summed (bars of the small case's test)."""
    n = 1 << 17
    pos, vel, mass = A.ic_mixed(n, 4)
    ctx.set_params(G=1.0, softening=2.5e-5, theta=0.0)
    ctx.set_state(pos, vel, mass)
    acc = ctx.forces(A.BH_GROUP)
    inter, _ = ctx.bh_stats()
    ref = ctx.forces(A.ALLPAIRS_FP64)
    scale = np.linalg.norm(ref, axis=1)
    err = np.linalg.norm(acc - ref, axis=1) / np.maximum(scale, np.median(scale))
    assert inter == n * (n - 1) and np.median(err) < 1e-6 and err.max() < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1025, 4095, 4096, 4097, 32768, 32769, 131073, 262144, 262145, 524288,
                               524289, 2097151])
@pytest.mark.parametrize("cells", ["spread", "few", "one"])
def test_sort_order_at_the_tiles_edges(ctx, n, cells):
    """(code, body) order against numpy where the tile, the kernel or the way to the digit starts changes, also with most
    or all keys equal."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(-1.0, 1.0, (n, 3)) * {"spread": 1.0, "few": 0.004, "one": 1e-9}[cells] + 1e-3
    ctx.set_params(G=1.0, softening=1e-2, theta=1.5, box=(1.0, 1.0, 1.0))
    ctx.set_state(pos, np.zeros_like(pos), np.ones(n))
    codes, _ = ctx.morton()
    ctx.forces(A.BH_GROUP, out=False)
    tree = ctx.tree()
    ref = np.lexsort((np.arange(n), codes))
    assert np.array_equal(tree["perm"], ref) and np.array_equal(tree["codes"], codes[ref])


@pytest.mark.gpu
@pytest.mark.parametrize("n,flags", [(65536, 0), (65537, 0), (262145, 0), (65536, A.PN1), (65537, A.PN1), (262145, A.PN1),
                                     (9000, A.PN1 | A.PN2)])
def test_wavefronts_per_group(ctx, orc, n, flags):
    """The oracle's lists and forces on both sides of the rule's lines (bars of the traversal's own tests)."""
    pos, vel, mass = A.ic_mixed(n, 5)
    box = orc.box_auto(pos)
    ctx.set_params(G=1.0, softening=2.5e-5, theta=0.7, c=30.0)
    ctx.set_state(pos, vel, mass)
    newton = ctx.forces(A.BH_GROUP)
    if not flags:
        ref, inter, visits = orc.bh_group(pos, mass, box, 0.7, soft=2.5e-5)
        assert ctx.bh_stats() == (inter, visits)
        scale = np.linalg.norm(ref, axis=1)
        err = np.linalg.norm(newton - ref, axis=1) / np.maximum(scale, np.median(scale))
        assert np.median(err) < 1e-6 and err.max() < 1e-4
        return
    ctx.set_params(G=1.0, softening=2.5e-5, theta=0.7, c=30.0, pn_flags=A.NEWTON | flags)
    both = ctx.forces(A.BH_GROUP)
    ref = orc.bh_group_pn(pos, vel, mass, box, 0.7, c=30.0, soft=2.5e-5, pn=A.NEWTON | flags)
    scale = np.linalg.norm(ref, axis=1)
    err = np.linalg.norm(both - newton - ref, axis=1)
    assert np.all(err <= 1e-9 * np.maximum(scale, np.median(scale)) + 1e-15 * np.abs(both).max())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 15, 16, 17, 16383, 16384, 16385, 131072, 131073, 147457, 1 << 20, (1 << 20) + 1,
                               (1 << 20) + 16400])
def test_group_starts_at_the_edges_of_chunks(ctx, orc, n):
    """The groups decide both counts of the lists and which nodes' moments are formed where."""
    pos, vel, mass = A.ic_mixed(n, 9)
    box = orc.box_auto(pos)
    ref = orc.build_tree(pos, vel, mass, box)
    ctx.set_params(G=1.0, softening=2.5e-5, theta=0.7)
    ctx.set_state(pos, vel, mass)
    ctx.forces(A.BH_GROUP, out=False)
    _, inter, visits = orc.bh_group(pos, mass, box, 0.7, soft=2.5e-5)
    assert ctx.bh_stats() == (inter, visits)
    tree = ctx.tree()
    for key in ("perm", "left", "right", "mass", "com"):
        assert np.array_equal(tree[key], ref[key]), key
