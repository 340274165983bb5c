"""Full CSG trees of height 4 to 7 with every leaf form, complements and infinite leaves among
their operands: every prim's GPU intersect equals the oracle's bit for bit, with single- and
double-precision roots. Trees this deep fill the walk's partial intersects and nest its
tranches beyond the entries it holds in registers, up to the capacities that end it."""
import numpy as np
import pytest

from oxr import abi
from oxr.csg import Foundry, box3, convexpolyhedron, halfspace, hyperboloid, phicut, translate, rotate_z_to

from test_gpu_parity import bits, random_rays
from test_gpu_random_csg import random_leaf

pytestmark = pytest.mark.gpu


def leaf(rng):
    k = int(rng.integers(0, 9))
    if k == 0:
        h = rng.uniform(15.0, 60.0, size=3)
        planes = np.zeros((6, 4))
        for a in range(3):
            planes[2 * a, a], planes[2 * a + 1, a] = 1.0, -1.0
            planes[2 * a, 3] = planes[2 * a + 1, 3] = h[a]
        t = convexpolyhedron(planes, [-h[0], -h[1], -h[2], h[0], h[1], h[2]])
        return t.moved(rotate_z_to(rng.normal(size=3))).moved(translate(*[float(x) for x in rng.uniform(-30, 30, size=3)]))
    if k == 1:
        return hyperboloid(float(rng.uniform(10, 40)), float(rng.uniform(20, 60)), -float(rng.uniform(20, 60)), float(rng.uniform(20, 60)))
    if k == 2:
        n = rng.normal(size=3)
        n /= np.linalg.norm(n)
        return random_leaf(rng) & halfspace(float(n[0]), float(n[1]), float(n[2]), float(rng.uniform(-20, 20)))
    if k == 3:
        return random_leaf(rng) & phicut(float(rng.uniform(0.0, 0.9)), float(rng.uniform(1.0, 1.9)))
    return random_leaf(rng)


def full_tree(rng, depth):
    if depth == 0:
        return leaf(rng)
    a, b = full_tree(rng, depth - 1), full_tree(rng, depth - 1)
    op = int(rng.integers(0, 3))
    return a | b if op == 0 else (a & b if op == 1 else a - b)


@pytest.mark.parametrize('fp64', [0, 1])
@pytest.mark.parametrize('depth', [2, 4, 5])
def test_deep_trees_bitexact(engine_mod, oracle_lib, depth, fp64):
    n = 10
    rng = np.random.default_rng(1000 * depth + fp64)
    f = Foundry()
    f.add_material('M', 1.0)
    b = f.boundary('M', None, None, 'M')
    f.begin_solid('deep')
    for _ in range(n):
        f.add_prim(full_tree(rng, depth) | box3(10.0), b)
    f.end_solid()
    f.add_instance(np.eye(4), 0)
    cfg = abi.default_config(fp64_roots=fp64)
    o = oracle_lib.Oracle(f.arrays(), f.physics(), cfg)
    print('deep CSG trees, depth', depth, 'fp64', fp64, 'nodes', len(f.arrays()['node']), flush=True)
    hits = 0
    with engine_mod.Engine(f.arrays(), f.physics(), cfg) as e:
        for p in range(n):
            rays = random_rays(rng, 2000, 100.0)
            gi, gv = e.intersect_prim(p, rays)
            oi, ov = o.intersect_prim(p, rays, 0)
            assert np.array_equal(gv, ov), (depth, p)
            assert np.array_equal(bits(gi), bits(oi)), (depth, p)
            hits += int(gv.sum())
    assert hits > 0
