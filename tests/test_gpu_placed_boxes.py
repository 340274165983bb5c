"""World boxes of placed prims formed from their leaves' shapes: rays that graze the turned
solids' silhouettes from inside to well outside, from far away, where a single-precision
quadric test may report a hit on a ray that passes the exact surface, find the hits of the
oracle's unculled loop in both BVH forms, bit for bit."""
import numpy as np
import pytest

from oxr import abi
from oxr.csg import Foundry, sphere, box3, zsphere, cylinder, scale, translate, rotate_z_to
from oxr.scenes import pmt_like_solid

from test_gpu_parity import bits

pytestmark = pytest.mark.gpu

# solid, its farthest surface from the axis of its placement (mm)
SOLIDS = {'bulb': (pmt_like_solid, 254.0), 'rod': (lambda: cylinder(20.0, -300.0, 200.0), 20.0),
          'lens': (lambda: zsphere(60.0, -20.0, 45.0).moved(scale(1.0, 1.6, 0.5)), 60.0),
          'ball': (lambda: sphere(30.0), 30.0), 'brick': (lambda: box3(80.0, 50.0, 30.0), 40.0)}


@pytest.mark.parametrize('name', sorted(SOLIDS))
def test_grazing_rays(engine_mod, oracle_lib, name):
    make, r = SOLIDS[name]
    rng = np.random.default_rng(len(name))
    f = Foundry()
    f.add_material('Air', 1.0)
    f.add_material('Glass', 1.5)
    f.begin_solid('r0')
    f.add_prim(sphere(6000.0), f.boundary('Air', None, None, 'Air'))
    f.end_solid()
    f.begin_solid('r1')
    f.add_prim(make(), f.boundary('Air', None, None, 'Glass'))
    f.end_solid()
    f.add_instance(np.eye(4), 0)
    centres = rng.uniform(-2500.0, 2500.0, size=(24, 3))
    for c in centres:
        f.add_instance(rotate_z_to(rng.normal(size=3)) @ translate(*c), 1)
    n = 40_000
    which = rng.integers(0, len(centres), size=n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    side = np.cross(d, rng.normal(size=(n, 3)))
    side /= np.linalg.norm(side, axis=1)[:, None]
    off = r * np.where(rng.uniform(size=n) < 0.7, rng.uniform(0.97, 1.01, size=n), rng.uniform(0.2, 1.6, size=n))
    rays = np.zeros((n, 2, 4), dtype=np.float32)
    rays[:, 0, :3] = centres[which] + off[:, None] * side - rng.uniform(400.0, 3000.0, size=n)[:, None] * d
    rays[:, 0, 3] = 0.05
    rays[:, 1, :3] = d
    rays[:, 1, 3] = 1e6
    g, p = f.arrays(), f.physics()
    cfg = abi.default_config()
    print('grazing rays', name, flush=True)
    want = oracle_lib.Oracle(g, p, cfg).trace(rays)
    iindex = bits(want)[:, 1, 2] >> 16
    assert (iindex != 0).mean() > 0.2          # the solids are hit, not only the world
    with engine_mod.Engine(g, p, cfg) as e:
        for bvh in (0, 1):
            e.set_tuning(bvh_mode=bvh)
            assert np.array_equal(bits(e.trace(rays)), bits(want)), (name, bvh)
