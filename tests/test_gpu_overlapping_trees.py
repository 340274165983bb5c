"""Prims whose trees share nodes at different places: a tree of seven nodes and one of three
begin inside a tree of fifteen, so each needs nodes of its own on the device with its own
links, behind those of the geometry. Every intersect, trace and photon equals the oracle's bit
for bit, with the nodes read in place and from their copy in LDS."""
import numpy as np
import pytest

from oxr import abi, gensteps as G
from oxr.csg import Foundry, box3, cylinder, rotate_z_to, scale, sphere, translate, zsphere

from test_gpu_parity import bits, random_rays

pytestmark = pytest.mark.gpu

UNION, INTERSECTION = 1, 2


def arrays():
    """Fifteen node records: operators 0 to 5, leaves 6 to 12 (record 6 at the third level of
    the large tree), zeros 13 and 14. Prims: the large tree, the one of records 3 to 9 twice,
    the one of records 5 to 7, the leaf of record 8, the large tree again."""
    f = Foundry()
    f.add_material('Air', 1.0)
    f.add_material('Glass', 1.5, absorption_length=2000.0, scattering_length=3000.0)
    b = f.boundary('Air', None, None, 'Glass')
    f.begin_solid('s')
    leaves = [box3(70.0), sphere(45.0).moved(translate(20.0, 5.0, -3.0)), cylinder(25.0, -80.0, 60.0).moved(rotate_z_to([1.0, 0.3, 0.2])),
              zsphere(60.0, -30.0, 40.0).moved(scale(1.0, 1.3, 0.8)), box3(50.0).moved(translate(-25.0, 10.0, 15.0)),
              sphere(38.0).moved(translate(-10.0, -30.0, 20.0)), cylinder(30.0, -40.0, 45.0).moved(translate(0.0, 25.0, 0.0))]
    for x in leaves:
        f.add_prim(x, b)
    f.end_solid()
    f.begin_solid('world')
    f.add_prim(sphere(600.0), f.boundary('Air', None, None, 'Air'))
    f.end_solid()
    f.add_instance(np.eye(4), 1)
    f.add_instance(rotate_z_to([0.3, -0.5, 0.8]) @ translate(40.0, -60.0, 30.0), 0)
    f.add_instance(translate(-250.0, 100.0, 20.0), 0)
    g = {k: v.copy() if isinstance(v, np.ndarray) else v for k, v in f.arrays().items()}
    leaf = g['node'].reshape(-1, 16)
    node = np.zeros((16, 16), dtype=np.float32)
    u = node.view(np.uint32)
    for k, op in enumerate((UNION, UNION, INTERSECTION, INTERSECTION, UNION, INTERSECTION)):
        u[k, 14] = op
    u[0, 0], u[3, 0], u[5, 0] = 15, 7, 3
    node[6:13] = leaf[:7]
    u[8, 15] |= 0x80000000            # a complement within the operands
    node[15] = leaf[7]
    u[:15, 6] = b
    prim = np.zeros((7, 16), dtype=np.float32)
    i = prim.view(np.int32)
    for k, (num, at) in enumerate([(15, 0), (7, 3), (7, 3), (3, 5), (1, 9), (15, 0)]):
        i[k, :2] = num, at
        prim[k, 8:14] = [-150.0] * 3 + [150.0] * 3
        i[k, 15] = k
    prim[6] = g['prim'].reshape(-1, 16)[7]
    i[6, 1], i[6, 15] = 15, 6
    solid = g['solid'].reshape(-1, 12)
    solid[0, 4:6] = 6, 0
    solid[1, 4:6] = 1, 6
    g['node'], g['prim'], g['solid'] = node.reshape(-1, 4, 4), prim.reshape(-1, 4, 4), solid.reshape(-1, 3, 4)
    return g, f.physics()


@pytest.mark.parametrize('fp64', [0, 1])
def test_intersects(engine_mod, oracle_lib, fp64):
    g, p = arrays()
    cfg = abi.default_config(fp64_roots=fp64)
    o = oracle_lib.Oracle(g, p, cfg)
    rng = np.random.default_rng(11)
    print('overlapping trees, fp64', fp64, flush=True)
    with engine_mod.Engine(g, p, cfg) as e:
        for k in range(7):
            rays = random_rays(rng, 4000, 110.0)
            gi, gv = e.intersect_prim(k, rays)
            oi, ov = o.intersect_prim(k, rays, 0)
            assert np.array_equal(gv, ov) and ov.sum() > 100, k
            assert np.array_equal(bits(gi), bits(oi)), k
        q = random_rays(rng, 8000, 300.0)
        q[:, 0, 3], q[:, 1, 3] = 0.05, 1e6
        for bvh in (0, 1):
            e.set_tuning(bvh_mode=bvh)
            assert np.array_equal(bits(e.trace(q)), bits(o.trace(q))), bvh


def test_photons(engine_mod, oracle_lib):
    g, p = arrays()
    gs = G.torch(np.array([3000, 1001]), pos=np.array([[40.0, -60.0, 30.0], [-200.0, 50.0, 0.0]]), wavelength=440.0,
                 type=G.T_POINT_ISOTROPIC)
    for fp64 in (0, 1):
        cfg = abi.default_config(max_bounce=20, fp64_roots=fp64)
        want = oracle_lib.Oracle(g, p, cfg).simulate(gs, seq=False)['photon']
        with engine_mod.Engine(g, p, cfg) as e:
            e.set_gensteps(gs)
            for stacks in (0, 1):
                for block in (64, 256):
                    e.set_tuning(block_size=block, csg_stack=stacks)
                    print('photons, fp64', fp64, 'block', block, 'nodes in LDS', e.info()['csg_in_lds'], flush=True)
                    assert e.info()['csg_in_lds'] == (1 if not fp64 else 0)
                    for form in (abi.OXR_FORM_PERSISTENT, abi.OXR_FORM_PLAIN):
                        e.launch(form)
                        assert np.array_equal(bits(e.photons()), bits(want)), (fp64, stacks, block, form)
