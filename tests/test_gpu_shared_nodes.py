"""Prims that share CSG nodes: two prims over one tree and one over a leaf inside it. The
device's nodes carry the links of one tree each, so the second tree needs a copy of its own;
every intersect and trace equals the oracle's bit for bit."""
import numpy as np
import pytest

from oxr import abi
from oxr.csg import Foundry, box3, sphere, cylinder, translate

from test_gpu_parity import bits, random_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fp64', [0, 1])
def test_shared_nodes(engine_mod, oracle_lib, fp64):
    f = Foundry()
    f.add_material('M', 1.0)
    b = f.boundary('M', None, None, 'M')
    f.begin_solid('shared')
    ball = sphere(60.0).moved(translate(15.0, 0.0, 0.0))
    for _ in range(4):
        f.add_prim((box3(80.0) - ball) | (cylinder(20.0, -90.0, 90.0) - sphere(35.0)), b)
    f.end_solid()
    f.add_instance(np.eye(4), 0)
    g = {k: v.copy() if isinstance(v, np.ndarray) else v for k, v in f.arrays().items()}
    prim = g['prim'].view(np.int32).reshape(4, -1)
    num, off = int(prim[0, 0]), int(prim[0, 1])
    assert num == 7
    prim[1, :2] = num, off           # the whole tree again
    prim[2, :2] = 1, off + 3         # its first leaf alone; prim 3 keeps its own tree
    cfg = abi.default_config(fp64_roots=fp64)
    o = oracle_lib.Oracle(g, f.physics(), cfg)
    rng = np.random.default_rng(9)
    print('shared nodes, fp64', fp64, flush=True)
    with engine_mod.Engine(g, f.physics(), cfg) as e:
        for p in range(4):
            rays = random_rays(rng, 3000, 110.0)
            gi, gv = e.intersect_prim(p, rays)
            oi, ov = o.intersect_prim(p, rays, 0)
            assert np.array_equal(gv, ov) and gv.sum() > 100, p
            assert np.array_equal(bits(gi), bits(oi)), p
        n = len(rays)
        q = rays.copy()
        q[:, 0, 3], q[:, 1, 3] = 0.05, 1e6
        assert np.array_equal(bits(e.trace(q)), bits(o.trace(q)))
